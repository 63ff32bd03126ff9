"""The filter, noise and lookup kernels (zh_field.hip) at the edges of their
strips, tiles and caches, against the oracle and the interpreter's bytes."""
import numpy as np
import pytest

import zosimos_amd as z
from oracle import color as C
from oracle import pipelines as PL

from gpu_util import run_both

pytestmark = pytest.mark.gpu

SB, SP, T = z.SampleBits, z.SampleParts, z.Transfer
LINEAR = z.Color(transfer=T.Linear)


def _image(kind, w, h, rng):
    """Descriptor, bytes and decoded FP64 colours of a random image."""
    if kind == "f32":
        v = rng.random((h, w, 4)).astype(np.float32)
        return z.Descriptor(w, h, z.Texel(SB.Float32x4, SP.RgbA), LINEAR), v, v.astype(np.float64)
    if kind == "f16":
        v = rng.random((h, w, 4)).astype(np.float16)
        return z.Descriptor(w, h, z.Texel(SB.Float16x4, SP.RgbA), LINEAR), v, v.astype(np.float64)
    top, dt, bits = (255, np.uint8, SB.UInt8x4) if kind == "u8" else (65535, np.uint16, SB.UInt16x4)
    raw = rng.integers(0, top + 1, (h, w, 4)).astype(dt)
    return z.Descriptor(w, h, z.Texel(bits, SP.RgbA), LINEAR), raw, raw.astype(np.float64) / top


# One column and one row, a partial group, a row past one workgroup's 1024
# columns, and enough rows for strips of more than one row on the whole chip
# (a strip boundary every 2 to 6 rows).
@pytest.mark.parametrize("w,h", [(1, 1), (1, 9), (7, 1), (5, 4), (1030, 3), (2051, 1601)])
@pytest.mark.parametrize("kind", ["u8", "f16", "f32", "u16"])
@pytest.mark.parametrize("direction", [z.Direction.Width, z.Direction.Height])
def test_box3_strips(ctx, kind, direction, w, h):
    """Sobel of a linear image (values in [-0.5, 0.5]): six products of f32
    colours sum within 6 ulps of 0.5 (4e-7), then the target's own rounding;
    the 8- and 16-bit targets clamp the negative half to 0."""
    d, raw, v = _image(kind, w, h, np.random.default_rng([w, h]))
    cmd = z.CommandBuffer()
    a = cmd.input(d)
    o, od = cmd.output(cmd.derivative(a, z.DerivativeMethod.Sobel, direction))
    out, exe = run_both(ctx, cmd, {a: d}, {a: raw.view(np.uint8).reshape(h, -1)}, {o: od})
    assert "field kernel" in exe.describe()
    want = PL.box3(v, PL.derivative_weights(z.DerivativeMethod.Sobel, width=direction == z.Direction.Width))
    got = out[o].reshape(-1).view(raw.dtype).reshape(h, w, 4)
    if kind in ("u8", "u16"):
        top = 255 if kind == "u8" else 65535
        code = np.rint(np.clip(want, 0, 1) * top).astype(np.int64)
        # u8 rounds to nearest, u16 truncates: within one code either way.
        assert np.abs(got.astype(np.int64) - code).max() <= 1
        assert np.all(got[..., 3] == top)
    else:
        step = 2.0 ** -12 if kind == "f16" else 0.0  # half an f16 ulp of values below 0.5
        assert np.all(np.abs(got.astype(np.float64) - want) <= 4e-7 + step)


@pytest.mark.parametrize("transfer", [T.Bt709, T.Bt470M, T.Bt601, T.Smpte240, T.Bt2020_10bit, T.Smpte2084, T.Srgb])
@pytest.mark.parametrize("bits", [SB.UInt8x4, SB.UInt16x4])
def test_box3_transfers(ctx, bits, transfer):
    """Derivatives of images with a transfer, every 8-bit code among them: the
    interpreter's bytes (run_both), NaN where it has them (SMPTE 240 has none
    between its segments, so there no zero weight may be skipped)."""
    w, h = 70, 37
    rng = np.random.default_rng(int(transfer))
    raw = rng.integers(0, 256, (h, w * z.BITS_BYTES[bits]), dtype=np.uint8)
    raw.reshape(-1)[:256] = np.arange(256)
    d = z.Descriptor(w, h, z.Texel(bits, SP.RgbA), z.Color(transfer=transfer))
    for method in (z.DerivativeMethod.Sobel, z.DerivativeMethod.Scharr3):
        cmd = z.CommandBuffer()
        a = cmd.input(d)
        v = cmd.derivative(a, method, z.Direction.Width)
        o, od = cmd.output(v)
        _, exe = run_both(ctx, cmd, {a: d}, {a: raw}, {o: od})
        assert "field kernel" in exe.describe()


# Octaves past the cached ones, cells smaller than a pixel (nothing fits the
# cache, or only the low octaves), several tiles with ragged edges, an octave
# count of 0; and images of so few tiles (under 1024) and so many corners that
# they stay on the interpreter.
@pytest.mark.parametrize("w,h,octaves,scale,kernel", [
    (2560, 410, 3, (280.0, 130.0), True), (2553, 415, 12, (70.0, 90.0), True), (2561, 401, 2, (150000.0, 80.0), True),
    (1600, 660, 5, (1200.0, 900.0), True), (2000, 520, 4, (1e6, 1e6), True), (3, 2, 0, (5.0, 5.0), True),
    (64, 16, 3, (7.0, 5.0), False), (131, 37, 12, (3.0, 8.0), False), (65, 17, 2, (4000.0, 3.0), False),
    (200, 50, 5, (150.0, 90.0), False), (70, 20, 4, (1e6, 1e6), False), (64, 16, 1, (7.0, 5.0), True),
    (331, 137, 3, (7.0, 5.0), True)])
def test_noise_cache(ctx, w, h, octaves, scale, kernel):
    """The noise's values are a fixed function of f32 arithmetic: bit-exact."""
    n = z.FractalNoise(octaves, 0.25, 0.75, scale)
    cmd = z.CommandBuffer()
    o, od = cmd.output(cmd.distribution_fractal_noise(z.Descriptor.rgba32f_linear(w, h), n))
    out, exe = run_both(ctx, cmd, {}, {}, {o: od})
    assert ("field kernel" in exe.describe()) == kernel
    want = PL.fractal_noise(w, h, octaves, n.initial_amplitude, n.amplitude_damping, scale).astype(np.float32)
    assert np.array_equal(out[o].view(np.float32).reshape(h, w, 4), want)


@pytest.mark.parametrize("ow,oh", [(1, 1), (9, 3), (301, 70)])
@pytest.mark.parametrize("kind", ["u8", "f16", "u16"])
def test_lookup(ctx, kind, ow, oh):
    """resize: the palette texel the rounded ramp selects, moved unchanged
    (linear codes and halves survive decode and encode)."""
    w, h = 50, 30
    d, raw, _ = _image(kind, w, h, np.random.default_rng([ow, oh]))
    cmd = z.CommandBuffer()
    a = cmd.input(d)
    o, od = cmd.output(cmd.resize(a, ow, oh))
    out, exe = run_both(ctx, cmd, {a: d}, {a: raw.view(np.uint8).reshape(h, -1)}, {o: od})
    assert "field kernel" in exe.describe()
    f = np.float32
    ramp = np.zeros((oh, ow, 4), f)
    ramp[..., 0] = ((np.arange(ow, dtype=f) + f(0.5)) / f(ow))[None, :]
    ramp[..., 1] = ((np.arange(oh, dtype=f) + f(0.5)) / f(oh))[:, None]
    ramp[..., 3] = 1.0
    ramp8 = (np.clip(ramp, 0, 1) * f(255.0)).astype(np.uint32).astype(f) / f(255.0)
    want = PL.palette_lookup(raw, ramp8, [1, 0, 0, 0], [0, 1, 0, 0])
    assert np.array_equal(out[o].reshape(-1).view(raw.dtype).reshape(oh, ow, 4), want)


@pytest.mark.parametrize("w,h", [(1, 1), (6, 3), (1031, 5)])
@pytest.mark.parametrize("bits,parts", [(SB.UInt8, SP.Luma), (SB.UInt8x3, SP.Rgb)])
def test_generator_rows_at_any_address(ctx, bits, parts, w, h):
    """Generated rows of 1- and 3-byte texels start at any byte: the ramp's
    truncated codes, linear transfer."""
    d = z.Descriptor(w, h, z.Texel(bits, parts), LINEAR)
    cmd = z.CommandBuffer()
    o, od = cmd.output(cmd.bilinear(d, z.Bilinear(u_max=(1.0, 0.0, 1.0, 1.0), v_max=(0.0, 1.0, 0.0, 0.0))))
    out, exe = run_both(ctx, cmd, {}, {}, {o: od})
    assert "field kernel" in exe.describe()
    f = np.float32
    u = np.broadcast_to(((np.arange(w, dtype=f) + f(0.5)) / f(w))[None, :], (h, w))
    v = np.broadcast_to(((np.arange(h, dtype=f) + f(0.5)) / f(h))[:, None], (h, w))
    want = np.stack([u, v, u], -1)[..., :1 if bits == SB.UInt8 else 3]
    exp = (want * f(255.0)).astype(np.uint32)
    assert np.array_equal(out[o].reshape(h, w, -1), exp.astype(np.uint8))
