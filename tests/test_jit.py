"""Planning of run-time kernels (no GPU): a flat pointwise chain without a
registered specialised kernel is marked for one compiled at run time, unless
ZH_PLAN_NO_JIT asks for the interpreter; registered chains keep their
kernels, and chains with operations the specialised bodies lack stay on the
interpreter."""
import ctypes
import itertools

import zosimos_amd as z
from zosimos_amd import workloads as W


def describe(cmd, flags=0):
    return z.Linker.from_included().compile(cmd).lower_to(None, flags).describe()


def test_unregistered_chain_is_compiled_at_run_time():
    wl = W.c2_reordered(64, 32)
    assert "[kernel jit#" in describe(wl.commands)
    assert "[kernel interp-inline]" in describe(wl.commands, z.PLAN_NO_JIT)
    # the same signature twice: one kernel id
    a = describe(W.c2_reordered(64, 32).commands).split("jit#")[1].split("]")[0]
    b = describe(W.c2_reordered(128, 16).commands).split("jit#")[1].split("]")[0]
    assert a == b


def srlab_chain(out):
    """SrLab2's encode of an RGBA8 image into half-float Lab, or of one with
    linear texels (no registered signature)."""
    d = z.Descriptor.rgba8_srgb(32, 32) if out == "registered" else z.Descriptor.rgba32f_linear(32, 32)
    cmd = z.CommandBuffer()
    cmd.output(cmd.color_convert(cmd.input(d), z.Color(model=z.ColorModel.SrLab2),
                                 z.Texel(z.SampleBits.Float16x4, z.SampleParts.LabA)))
    return cmd


def test_registered_and_unsupported_chains():
    assert "[kernel c2_over" in describe(W.c2(64, 32).commands)
    # SrLab2's encode is registered for RGBA8, and compiled for other texels
    assert "[kernel srlab_enc_s8h]" in describe(srlab_chain("registered"))
    assert "[kernel jit#" in describe(srlab_chain("linear"))
    # no specialised body takes a channel apart
    d = z.Descriptor.rgba8_srgb(32, 32)
    cmd = z.CommandBuffer()
    a, b = cmd.input(d), cmd.input(d)
    cmd.output(cmd.inject(a, z.ColorChannel.G, cmd.extract(b, z.ColorChannel.R)))
    text = describe(cmd)
    assert " channel " in text and "[kernel interp-inline]" in text and "jit#" not in text, text


def test_tag_names_the_kernel_that_runs():
    """An unregistered conversion of in-line formats without run-time kernels
    runs on the any-format kernel, not the interpreter."""
    src = z.Descriptor.rgba32f_linear(33, 7)
    cmd = z.CommandBuffer()
    a = cmd.input(src)
    cmd.output(cmd.color_convert(a, z.Color(primaries=z.Primaries.DisplayP3),
                                 z.Texel(z.SampleBits.UInt8x4, z.SampleParts.BgrA)))
    assert "[kernel jit#" in describe(cmd)
    text = describe(cmd, z.PLAN_NO_JIT)
    assert "[any-format kernel]" in text and "interp" not in text, text


def test_unregistered_warp_form_is_compiled_at_run_time():
    d = z.Descriptor(200, 120, W.RGBA16F, W.P3_LINEAR)
    cmd = z.CommandBuffer()
    a = cmd.input(d)
    canvas = cmd.solid_rgba(z.Descriptor(300, 180, W.RGBA16F, W.P3_LINEAR), (0, 0, 0, 0))
    r = cmd.affine(canvas, z.Affine.new(z.AffineSample.BiLinear).rotate(0.3), a)
    cmd.output(cmd.color_convert(r, z.Color.SRGB, W.RGBA8))
    assert "post[unpremul mat3 store#1] [kernel jitw#" in describe(cmd)
    assert "jitw#" not in describe(cmd, z.PLAN_NO_JIT)
    # axis-aligned maps pick the separable form
    cmd2 = z.CommandBuffer()
    a2 = cmd2.input(d)
    c2 = cmd2.solid_rgba(z.Descriptor(300, 180, W.RGBA16F, W.P3_LINEAR), (0, 0, 0, 0))
    r2 = cmd2.affine(c2, z.Affine.new(z.AffineSample.BiLinear).scale(1.5, 1.5), a2)
    cmd2.output(cmd2.color_convert(r2, z.Color.SRGB, W.RGBA8))
    assert "_sep]" in describe(cmd2).split("jitw#")[1]
    assert "_sep_lds]" in describe(cmd2, z.PLAN_STAGED).split("jitw#")[1]


def _warp_grid(tiles, resident, cus=256, per_cu=0, persistent=0, layers=0):
    blocks, run = ctypes.c_uint32(), ctypes.c_uint32()
    z._abi.lib().zh_warp_grid(*map(ctypes.c_uint32, (tiles, resident, cus, per_cu)), ctypes.c_int(persistent),
                              ctypes.c_uint32(layers), ctypes.byref(blocks), ctypes.byref(run))
    return blocks.value, run.value


def test_warp_grids_cover_their_tiles():
    """Runs of tiles for grids past the resident one: every tile in one run, no
    empty workgroup."""
    for resident, layers in itertools.product((1, 2, 3, 5, 7), (0, 1, 2, 8)):
        for tiles in (1, 255, 256 * resident, 256 * resident + 1, 8160, 100_003, 10_000_019):
            blocks, run = _warp_grid(tiles, resident, layers=layers)
            if tiles <= 256 * resident:
                assert run == 0 and blocks == tiles
            else:
                assert 1 <= run <= 8 and (blocks - 1) * run < tiles <= blocks * run
    # tables and one layer: two tiles a run
    assert [_warp_grid(8160, 5, layers=n)[1] for n in (0, 1, 2)] == [1, 2, 1]
    assert _warp_grid(100_000, 6, per_cu=2) == (512, 0)
    assert _warp_grid(100_000, 6, persistent=1) == (1536, 0)
