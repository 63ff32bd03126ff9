"""The texel-moving nearest kernel (zh_move.hip) at tile edges, for stacked
and partly outside paints, against a numpy restatement of the FP64 maps and
the interpreter's bytes."""
import math

import numpy as np
import pytest

import zosimos_amd as z
from oracle import pipelines as PL
from zosimos_amd import workloads as W

from gpu_util import run_both

pytestmark = pytest.mark.gpu

SB, SP, T = z.SampleBits, z.SampleParts, z.Transfer
KINDS = {"u8": (z.Texel(SB.UInt8x4, SP.RgbA), z.Color.SRGB, np.uint8),
         "bgra8": (z.Texel(SB.UInt8x4, SP.BgrA), z.Color(transfer=T.Linear), np.uint8),
         "f16": (z.Texel(SB.Float16x4, SP.RgbA), z.Color(transfer=T.Linear), np.float16),
         "f32": (z.Texel(SB.Float32x4, SP.RgbA), z.Color(transfer=T.Linear), np.float32)}


def _image(kind, w, h, seed, pad=0):
    tex, color, dt = KINDS[kind]
    rng = np.random.default_rng(seed)
    v = rng.integers(0, 256, (h, w, 4)).astype(dt) if dt == np.uint8 else rng.normal(0, 3, (h, w, 4)).astype(dt)
    d = z.Descriptor(w, h, tex, color, w * tex.bytes + pad if pad else 0)
    return d, v


def _bytes(v):
    return np.ascontiguousarray(v).view(np.uint8).reshape(v.shape[0], -1)


@pytest.mark.parametrize("w,h,fw,fh,pad", [(1, 1, 1, 1, 0), (64, 16, 63, 15, 0), (65, 17, 65, 16, 16), (200, 37, 8, 36, 4)])
@pytest.mark.parametrize("kind", list(KINDS))
def test_inscribe_moves_bytes(ctx, kind, w, h, fw, fh, pad):
    """A foreground over a background's corner, and a smaller one over both:
    every byte moved as it is (pads 16-byte aligned or only 4)."""
    (db, vb), (df, vf) = _image(kind, w, h, 1, pad), _image(kind, fw, fh, 2)
    gw, gh = max(1, fw // 2), max(1, fh // 2)
    dg, vg = _image(kind, gw, gh, 3)
    cmd = z.CommandBuffer()
    b, f, g = cmd.input(db), cmd.input(df), cmd.input(dg)
    v = cmd.inscribe(cmd.inscribe(b, z.Rectangle(0, 0, fw, fh), f), z.Rectangle(0, 0, gw, gh), g)
    o, od = cmd.output(v)
    out, exe = run_both(ctx, cmd, {b: db, f: df, g: dg}, {b: _bytes(vb), f: _bytes(vf), g: _bytes(vg)}, {o: od})
    want = vb.copy()
    # Rectangle::normalize takes max_y = y + width: the quad of a paint is as
    # tall as the rectangle is wide, cut at the target.
    for img, iw, ih in ((vf, fw, fh), (vg, gw, gh)):
        qh = iw
        ys = (np.arange(h) + 0.5) * ih / qh
        rows = ys < ih
        want[rows, :iw] = img[np.floor(ys[rows]).astype(int)]
    if w > 1 or h > 1:
        assert "move kernel" in exe.describe()
    assert np.array_equal(out[o], _bytes(want))


@pytest.mark.parametrize("degrees,scale", [(0.0, 1.0), (33.0, 0.9), (90.0, 2.5), (180.0, 0.1)])
@pytest.mark.parametrize("kind", ["u8", "f32"])
def test_nearest_affine_moves_texels(ctx, kind, degrees, scale):
    """A rotated and scaled nearest placement: the texel at the floor of the
    FP64 inverse of the pixel centre where that lies inside the source."""
    w, h, fw, fh = 131, 70, 40, 25
    (db, vb), (df, vf) = _image(kind, w, h, 4), _image(kind, fw, fh, 5)
    aff = W.about_centre(fw, fh, scale, math.radians(degrees), z.AffineSample.Nearest, out_wh=(w, h))
    cmd = z.CommandBuffer()
    b, f = cmd.input(db), cmd.input(df)
    o, od = cmd.output(cmd.affine(b, aff, f))
    out, exe = run_both(ctx, cmd, {b: db, f: df}, {b: _bytes(vb), f: _bytes(vf)}, {o: od})
    assert "move kernel" in exe.describe()
    got = out[o].reshape(h, w, -1)
    m = np.array(np.float32(aff.transformation), np.float64).reshape(3, 3)
    ys, xs = np.mgrid[0:h, 0:w]
    p = np.linalg.inv(m) @ np.stack([xs.ravel() + 0.5, ys.ravel() + 0.5, np.ones(w * h)])
    u, v = p[0].reshape(h, w), p[1].reshape(h, w)
    inside = (u >= 0) & (u < fw) & (v >= 0) & (v < fh)
    iu, iv = np.clip(np.floor(u).astype(int), 0, fw - 1), np.clip(np.floor(v).astype(int), 0, fh - 1)
    want = np.where(inside[..., None], vf[iv, iu].reshape(h, w, 4), vb)
    # Pixels whose centre maps within 1e-4 texel of a texel's edge may round to
    # either side (the quad's corners are f32).
    edge = (np.abs(u - np.rint(u)) < 1e-4) | (np.abs(v - np.rint(v)) < 1e-4)
    same = np.all(got == _bytes(want).reshape(h, w, -1), axis=-1)
    assert np.all(same | edge)


@pytest.mark.parametrize("w,h,rect", [(70, 33, (10, 5, 45, 30)), (64, 48, (8, 4, 40, 28))])
def test_crop_moves_texels(ctx, w, h, rect):
    """crop stretches the selection over an output of the source's size."""
    d, v = _image("u8", w, h, 6)
    cmd = z.CommandBuffer()
    a = cmd.input(d)
    o, od = cmd.output(cmd.crop(a, z.Rectangle(*rect)))
    out, exe = run_both(ctx, cmd, {a: d}, {a: _bytes(v)}, {o: od})
    assert "move kernel" in exe.describe()
    want = PL.crop(v.astype(np.float64), rect)
    assert np.array_equal(out[o].reshape(h, w, 4), want.astype(np.uint8))
