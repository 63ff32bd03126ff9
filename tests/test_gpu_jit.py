"""Kernels compiled at run time (zh_jit.cpp): a pointwise chain with no
registered specialised kernel -- C2's operations with the 'over' moved
first -- gets the specialised body compiled for its signature with hiprtc.
Its results are checked against the FP64 oracle and against the general
interpreter (ZH_PLAN_NO_JIT), alone and as a batch of ragged images run by
one launch, and inside a captured graph."""
import numpy as np
import pytest

import zosimos_amd as z
from zosimos_amd import workloads as W
from oracle import pipelines as PL

from gpu_util import compare_u8, report, run

pytestmark = pytest.mark.gpu


def test_unregistered_chain_runs_a_compiled_kernel(ctx):
    w, h = 320, 180
    wl = W.c2_reordered(w, h, seed=4)
    host = wl.make_inputs()
    (o, od), = wl.outputs.items()
    out, exe = run(ctx, wl.commands, wl.inputs, host, wl.outputs)
    text = exe.describe()
    assert "[kernel jit#" in text and "unavailable" not in text, text
    report("jit_compile", lines=[l for l in text.splitlines() if l.startswith("jit#")])
    src_r, layer_r = list(wl.inputs)
    lin, want = PL.c2_reordered(PL.u8_image(host[src_r], w, h), PL.f16_image(host[layer_r], w, h))
    mr, ma, exact = compare_u8("jit_c2_reordered", out[o], want, alpha_ok=want[..., 3] > 0)
    assert mr <= 1 and ma <= 1 and exact > 0.99
    interp, exe2 = run(ctx, wl.commands, wl.inputs, host, wl.outputs, flags=z.PLAN_NO_JIT)
    assert "interp-inline" in exe2.describe()
    diff = np.abs(out[o].astype(int) - interp[o].astype(int))
    report("jit_vs_interpreter", max_code_diff=int(diff.max()), equal=float((diff == 0).mean()))
    assert diff.max() <= 1


def test_compiled_kernel_batch_of_ragged_images(ctx):
    """Five images of the signature: one launch of the compiled batch kernel
    (one chunk of 1,024 pixels after the other; test_gpu_spec_chunks.py has the
    longer ones), each image within 1 code of its interpreter result."""
    sizes = [(1, 1), (7, 5), (129, 127), (300, 61), (16385, 2)]
    cmd = z.CommandBuffer()
    regs, inputs, host = [], {}, {}
    rng = np.random.default_rng(9)
    for w, h in sizes:
        d8 = z.Descriptor.rgba8_srgb(w, h)
        dl = z.Descriptor(w, h, W.RGBA16F, W.P3_LINEAR)
        a, b = cmd.input(d8), cmd.input(dl)
        p3 = cmd.color_convert(a, W.P3_LINEAR, W.RGBA16F)
        over = cmd.blend(p3, z.Rectangle(0, 0, w, h), b)
        lab = cmd.oklab_adjust(cmd.color_convert(over, z.Color.OKLAB, W.LABA16F), chroma=1.2, hue_rad=0.0)
        o, od = cmd.output(cmd.color_convert(cmd.color_convert(lab, W.P3_LINEAR, W.RGBA16F), W.P3_SRGB, W.RGBA8))
        inputs[a], inputs[b] = d8, dl
        host[a] = W.random_rgba8(rng, w, h)
        host[b] = W.random_rgba16f(rng, w, h)
        regs.append((a, b, o, od, w, h))
    outputs = {o: od for (_, _, o, od, _, _) in regs}
    out, exe = run(ctx, cmd, inputs, host, outputs)
    text = exe.describe()
    assert "[kernel jit#" in text and "over 5 stages" in text, text
    interp, _ = run(ctx, cmd, inputs, host, outputs, flags=z.PLAN_NO_JIT)
    for (a, b, o, od, w, h) in regs:
        lin, want = PL.c2_reordered(PL.u8_image(host[a], w, h), PL.f16_image(host[b], w, h))
        mr, ma, exact = compare_u8(f"jit_batch_{w}x{h}", out[o], want, alpha_ok=want[..., 3] > 0)
        assert mr <= 1 and ma <= 1
        assert np.abs(out[o].astype(int) - interp[o].astype(int)).max() <= 1


def test_compiled_kernel_inside_a_graph(ctx):
    """The compiled kernel between two other launches, captured once and
    replayed: every replay equals the eager program."""
    w, h = 256, 64
    wl = W.c2_reordered(w, h, seed=6)
    cmd = wl.commands
    (o, od), = wl.outputs.items()
    extra, extra_d = cmd.output(cmd.crop(list(wl.inputs)[0], z.Rectangle(0, 0, 64, 32)))
    host = wl.make_inputs()
    outputs = dict(wl.outputs)
    outputs[extra] = extra_d
    prog = z.Linker.from_included().compile(cmd)
    exe, eager = prog.lower_to(ctx), prog.lower_to(ctx, z.PLAN_NO_GRAPH)
    ins = {r: ctx.image(d) for r, d in wl.inputs.items()}
    for r, img in ins.items():
        img.upload(host[r])
    outs = {r: ctx.image(d) for r, d in outputs.items()}
    refs = {r: ctx.image(d) for r, d in outputs.items()}
    for _ in range(3):
        exe.launch(ins, outs)
        eager.launch(ins, refs)
        ctx.sync()
        for r in outs:
            assert np.array_equal(outs[r].download(), refs[r].download())
    g = exe.graph_info()
    report("jit_graph", **g)
    assert g["state"] == "captured" and g["replays"] >= 2


def test_unregistered_warp_form_runs_a_compiled_kernel(ctx):
    """A rotated RGBA16F layer composited onto a transparent canvas and
    converted from Display-P3 to sRGB: a post program (un-premultiply, matrix,
    store) no registered warp kernel has.  The compiled warp kernel against
    the FP64 oracle and the resample interpreter, alone and as a batch of two
    images (one launch)."""
    from oracle import color as C
    rng = np.random.default_rng(12)
    cmd = z.CommandBuffer()
    regs, host = [], {}
    for w, h, ow, oh in [(200, 120, 260, 200), (97, 64, 150, 101)]:
        d = z.Descriptor(w, h, W.RGBA16F, W.P3_LINEAR)
        a = cmd.input(d)
        canvas = cmd.solid_rgba(z.Descriptor(ow, oh, W.RGBA16F, W.P3_LINEAR), (0, 0, 0, 0))
        aff = z.Affine.new(z.AffineSample.BiLinear).rotate(0.3).shift(40.0, 10.0)
        r = cmd.affine(canvas, aff, a)
        o, od = cmd.output(cmd.color_convert(r, z.Color.SRGB, W.RGBA8))
        host[a] = W.random_rgba16f(rng, w, h)
        regs.append((a, d, o, od, aff, w, h, ow, oh))
    inputs = {a: d for (a, d, *_rest) in regs}
    outputs = {o: od for (_a, _d, o, od, *_rest) in regs}
    out, exe = run(ctx, cmd, inputs, host, outputs)
    text = exe.describe()
    assert "[kernel jitw#" in text and "over 2 stages" in text and "unavailable" not in text, text
    interp, exe2 = run(ctx, cmd, inputs, host, outputs, flags=z.PLAN_NO_JIT)
    assert "jitw#" not in exe2.describe()
    m709 = C.convert_matrix(7, 3, 5)
    for (a, d, o, od, aff, w, h, ow, oh) in regs:
        src = PL.f16_image(host[a], w, h)
        res = C.unpremultiply(C.bilinear_affine(C.premultiply(src), PL.mat_f32(aff.transformation), (oh, ow)))
        want = C.encode_u8(PL.apply3(m709, res), 5)
        mr, ma, exact = compare_u8(f"jitw_{w}x{h}", out[o], want, alpha_ok=res[..., 3] > 0.02)
        assert mr <= 1 and ma <= 1 and exact > 0.99
        diff = np.abs(out[o].astype(int) - interp[o].astype(int))
        report(f"jitw_vs_interpreter_{w}x{h}", max_code_diff=int(diff.max()), equal=float((diff == 0).mean()))
        assert diff.max() <= 1


@pytest.mark.parametrize("degrees", [0.0, 25.0])
def test_two_half_float_sources_hold_their_registers(ctx, degrees):
    """'over' of two RGBA16F images under an affine map, alone and as a batch:
    the compiled kernels (separable and general maps) spill no register, and
    each result is within one f16 ulp of the FP64 oracle (1e-6 absolute near
    zero)."""
    from oracle import color as C
    rng = np.random.default_rng(21)
    for sizes in ([(130, 70)], [(130, 70), (64, 33)]):
        cmd, inputs, host, outputs, want = z.CommandBuffer(), {}, {}, {}, {}
        for w, h in sizes:
            d = z.Descriptor.rgba16f_linear(w, h)
            a, b = cmd.input(d), cmd.input(d)
            ab = cmd.blend(a, z.Rectangle(0, 0, w, h), b)
            aff = W.about_centre(w, h, 0.8, np.deg2rad(degrees))
            o, od = cmd.output(cmd.affine(cmd.solid_rgba(d, (0, 0, 0, 0)), aff, ab))
            for r in (a, b):
                inputs[r], host[r] = d, W.random_rgba16f(rng, w, h)
            outputs[o] = od
            A, B = (C.premultiply(PL.f16_image(host[r], w, h)) for r in (a, b))
            want[o] = C.unpremultiply(C.bilinear_affine(C.over(B, A), PL.mat_f32(aff.transformation), (h, w)))
        out, exe = run(ctx, cmd, inputs, host, outputs)
        text = exe.describe()
        assert "\njitw#" in text and "unavailable" not in text, text
        assert "scratch" not in text, text
        for o, v in want.items():
            got = np.asarray(out[o]).reshape(-1).view(np.float16).reshape(v.shape)
            ulp = np.abs(got.view(np.int16).astype(int) - C.encode_f16(v).view(np.int16).astype(int))
            ulp = np.where(np.abs(got.astype(np.float64) - v) <= 1e-6, 0, ulp)
            assert np.where(v[..., 3:] > 1e-3, ulp, 0).max() <= 1


@pytest.mark.parametrize("degrees", [0.0, 12.0])
@pytest.mark.parametrize("texel,w,h,few", [
    ("f16", 63, 15, True), ("f16", 400, 300, True), ("f16", 1024, 256, True), ("f16", 1025, 256, False),
    ("f32", 63, 15, False), ("f32", 1025, 256, False), ("f32", 1400, 1400, False), ("u8", 400, 300, False)])
def test_compiled_form_of_few_tiles(ctx, texel, w, h, few, degrees):
    """Four layers through a compiled form: up to one tile per compute unit
    (256) of half floats the kernel without a choice of path runs, else the
    form's other (floats have only kernels without one); within 1 code of the FP64
    oracle (colour where alpha is above 0.02)."""
    from oracle import color as C
    rng = np.random.default_rng([w, h])
    cmd = z.CommandBuffer()
    tex, color = {"f16": (W.RGBA16F, W.P3_LINEAR), "f32": (z.Descriptor.rgba32f_linear(1, 1).texel, W.P3_LINEAR),
                  "u8": (W.RGBA8, W.P3_SRGB)}[texel]
    d = z.Descriptor(w, h, tex, color)
    acc = cmd.solid_rgba(d, (0, 0, 0, 0))
    inputs, host, want = {}, {}, np.zeros((h, w, 4))
    for k in range(4):
        a = cmd.input(d)
        inputs[a] = d
        if texel == "u8":
            host[a] = W.random_rgba8(rng, w, h)
            src = C.decode_u8(PL.u8_image(host[a], w, h), 5)
        else:
            host[a] = W.random_rgba16f(rng, w, h)
            src = PL.f16_image(host[a], w, h)
            if texel == "f32":
                host[a] = src.astype(np.float32).view(np.uint8).reshape(-1)
        aff = W.about_centre(w, h, 0.6 + 0.3 * k, np.deg2rad(degrees * k))
        acc = cmd.affine(acc, aff, a)
        want = C.over(C.bilinear_affine(C.premultiply(src), PL.mat_f32(aff.transformation), (h, w)), want)
    o, od = cmd.output(cmd.color_convert(acc, z.Color.SRGB, W.RGBA8))
    out, exe = run(ctx, cmd, inputs, host, {o: od})
    text = exe.describe()
    assert "[kernel jitw#" in text and ("kernel for few" in text) == few, text
    assert "scratch" not in text, text
    straight = C.unpremultiply(want)
    codes = C.encode_u8(PL.apply3(C.convert_matrix(7, 3, 5), straight), 5)
    mr, ma, _ = compare_u8(f"jitw_few_{texel}_{w}x{h}_{degrees}", out[o], codes, alpha_ok=straight[..., 3] > 0.02)
    assert mr <= 1 and ma <= 1


@pytest.mark.parametrize("w,h", [(5, 3), (257, 130)])
def test_compiled_srlab2_chain(ctx, w, h):
    """SrLab2 of linear RGBA32F texels into half-float and float Lab (no
    registered signature): compiled, the interpreter's bytes, and within 2e-5 of
    the FP64 oracle's L, a, b (f16 targets: half an f16 ulp of values below 2,
    2^-11, on top)."""
    from oracle import color as C
    rng = np.random.default_rng([w, h])
    v = rng.random((h, w, 4)).astype(np.float32)
    v.reshape(-1)[:8] = [0, 0, 0, 1, 1, 1, 1, 1]
    for bits, tol in ((z.SampleBits.Float16x4, 2e-5 + 2.0 ** -11), (z.SampleBits.Float32x4, 2e-5)):
        d = z.Descriptor.rgba32f_linear(w, h)
        cmd = z.CommandBuffer()
        a = cmd.input(d)
        o, od = cmd.output(cmd.color_convert(a, z.Color.SRLAB2_D65, z.Texel(bits, z.SampleParts.LabA)))
        host = {a: v.view(np.uint8).reshape(h, -1)}
        out, exe = run(ctx, cmd, {a: d}, host, {o: od})
        text = exe.describe()
        assert "[kernel jit#" in text and "unavailable" not in text, text
        ref, _ = run(ctx, cmd, {a: d}, host, {o: od}, flags=z.PLAN_INTERPRETER)
        assert np.array_equal(out[o], ref[o])
        dt = np.float16 if bits == z.SampleBits.Float16x4 else np.float32
        got = np.asarray(out[o]).reshape(-1).view(dt).reshape(h, w, 4).astype(np.float64)
        assert np.abs(got[..., :3] - C.rgb_to_srlab2(v[..., :3])).max() <= tol


@pytest.mark.parametrize("source", ["s8", "l8", "f16", "f32"])
@pytest.mark.parametrize("target", ["s8", "f16", "f32"])
def test_srlab2_after_an_over_keeps_the_interpreters_bytes(ctx, source, target):
    """'over' of two layers, to SrLab2 and back, alone and as a batch of two: the
    chains that ran on the interpreter before they were compiled give its bytes."""
    tex = {"s8": (W.RGBA8, z.Color.SRGB), "l8": (W.RGBA8, z.Color(transfer=z.Transfer.Linear)),
           "f16": (W.RGBA16F, z.Color(transfer=z.Transfer.Linear)),
           "f32": (z.Descriptor.rgba32f_linear(1, 1).texel, z.Color(transfer=z.Transfer.Linear))}
    rng = np.random.default_rng(31)
    for sizes in ([(257, 130)], [(257, 130), (61, 67)]):
        cmd, inputs, host, outputs = z.CommandBuffer(), {}, {}, {}
        for w, h in sizes:
            d = z.Descriptor(w, h, *tex[source])
            linear = []
            for _ in range(2):
                a = cmd.input(d)
                inputs[a] = d
                v = rng.random((h, w * 4))
                host[a] = {"f16": v.astype(np.float16), "f32": v.astype(np.float32)}.get(
                    source, (v * 256).astype(np.uint8)).view(np.uint8)
                linear.append(cmd.color_convert(a, z.Color(transfer=z.Transfer.Linear), W.RGBA16F))
            v = cmd.blend(linear[0], z.Rectangle(0, 0, w, h), linear[1])
            lab = cmd.color_convert(v, z.Color.SRLAB2_D65, W.LABA16F)
            o, od = cmd.output(cmd.color_convert(lab, tex[target][1], tex[target][0]))
            outputs[o] = od
        out, exe = run(ctx, cmd, inputs, host, outputs)
        text = exe.describe()
        assert "[kernel jit#" in text and "unavailable" not in text, text
        ref, _ = run(ctx, cmd, inputs, host, outputs, flags=z.PLAN_INTERPRETER)
        for o in outputs:
            assert np.array_equal(out[o], ref[o])
