"""The any-format pointwise kernels (zh_any.hip) at the sizes where a group,
a row or a table can go wrong, against the oracle's restatement of
stage.frag."""
import numpy as np
import pytest

import zosimos_amd as z
from oracle import color as C
from oracle import stage as S

from gpu_util import report, run_both

pytestmark = pytest.mark.gpu

SB, SP, T = z.SampleBits, z.SampleParts, z.Transfer
F32 = z.Texel(SB.Float32x4, SP.RgbA)
LINEAR = z.Color(transfer=T.Linear)

FORMATS = [(SB.UInt8, SP.Luma, T.Srgb), (SB.UInt233, SP.Rgb, T.Linear), (SB.UInt565, SP.Bgr, T.Srgb),
           (SB.UInt4x4, SP.ARgb, T.Linear), (SB.UInt8x2, SP.LumaA, T.Srgb), (SB.UInt8x3, SP.Rgb, T.Srgb),
           (SB.UInt8x4, SP.ABgr, T.Bt709), (SB.UInt1010102, SP.ARgb, T.Bt2020_10bit),
           (SB.UInt2101010, SP.RgbA, T.Bt601), (SB.UInt16, SP.R, T.Linear), (SB.UInt16x2, SP.LumaA, T.Srgb),
           (SB.UInt16x4, SP.RgbA, T.Srgb), (SB.UInt16x3, SP.Rgb, T.Linear)]


def _texels(bits, n, seed):
    """n random texels as (n, bytes) plus their 32-bit codes where they have one."""
    raw = np.random.default_rng(seed).integers(0, 256, (n, z.BITS_BYTES[bits]), dtype=np.uint8)
    pad = np.zeros((n, 4), np.uint8)
    pad[:, :min(4, raw.shape[1])] = raw[:, :4]
    return raw, pad.view(np.uint32).ravel()


def _decoded(bits, parts, transfer, raw, codes):
    if bits in (SB.UInt16x3, SB.UInt16x4):
        v = np.ones((raw.shape[0], 4), np.float32)
        ch = raw.shape[1] // 2
        v[:, :ch] = raw.view(np.uint16).reshape(-1, ch).astype(np.float32) / np.float32(65535.0)
        out = v.astype(np.float64)
        if transfer == T.Srgb:
            out[:, :3] = C.eo_srgb(out[:, :3])
        return out
    return S.stage_decode(codes, bits, parts, transfer)


def _pitch(w, bpp, pad):
    """Row bytes: a multiple of 4 for a positive pad, and for a negative one the
    odd number of texels that leaves rows of 1-, 2-, 3- and 6-byte texels at
    every address their size allows."""
    return 0 if not pad else (w * bpp + pad + 3) // 4 * 4 if pad > 0 else (w | 1) * bpp - 2 * pad * bpp


# Rows of 1-9 texels (partial groups only, one whole group, a whole and a
# partial one), a row past one workgroup, and a padded pitch.
@pytest.mark.parametrize("w,h,pad", [(1, 1, 0), (3, 5, 0), (4, 2, 12), (7, 3, 4), (9, 1, 0), (1031, 2, 0), (1029, 3, 20),
                                     (7, 5, -1), (1024, 5, -1), (1027, 3, -2)])
@pytest.mark.parametrize("bits,parts,transfer", FORMATS)
def test_any_format_conversion(ctx, bits, parts, transfer, w, h, pad):
    """Decode to RGBA32F (2-D for a padded pitch, flat otherwise), then encode
    the decoded values back (both the interpreter's bytes): bit-exact for linear transfers; a transfer is
    compared within the accuracy of two pow implementations (a few f32 ulps
    through an exponent of at most 2.4: 4e-6 relative, 1e-6 absolute)."""
    bpp = z.BITS_BYTES[bits]
    raw, codes = _texels(bits, w * h, [bits, parts, w, h])
    pitch = _pitch(w, bpp, pad)
    src = z.Descriptor(w, h, z.Texel(bits, parts), z.Color(transfer=transfer), pitch)
    cmd = z.CommandBuffer()
    a = cmd.input(src)
    o, od = cmd.output(cmd.color_convert(a, LINEAR, F32))
    out, exe = run_both(ctx, cmd, {a: src}, {a: raw.reshape(h, w * bpp)}, {o: od})
    assert "any-format kernel" in exe.describe()
    got = out[o].view(np.float32).reshape(-1, 4)
    want = _decoded(bits, parts, transfer, raw, codes)
    if transfer == T.Linear:
        assert np.array_equal(got, want.astype(np.float32))
    else:
        assert np.all(np.abs(got - want) <= 4e-6 * np.abs(want) + 1e-6)
    # Padded rows here too: the stores of the tight output then start at every
    # address a row of its texels can.
    cmd = z.CommandBuffer()
    f32 = z.Descriptor(w, h, F32, LINEAR, w * 16 + 16 if pad else 0)
    a = cmd.input(f32)
    o, od = cmd.output(cmd.color_convert(a, src.color, src.texel))
    out, exe = run_both(ctx, cmd, {a: f32}, {a: got.view(np.uint8).reshape(h, w * 16)}, {o: od})
    assert "any-format kernel" in exe.describe()
    if bits in (SB.UInt16x3, SB.UInt16x4) or transfer != T.Linear:
        return
    pad4 = np.zeros((w * h, 4), np.uint8)
    pad4[:, :bpp] = out[o].reshape(w * h, bpp)
    mask = np.uint32(0xffffffff) if bpp >= 4 else np.uint32((1 << (8 * bpp)) - 1)
    assert np.array_equal(pad4.view(np.uint32).ravel(), S.stage_encode(want, bits, parts, transfer) & mask)


@pytest.mark.parametrize("w,h,pad", [(2, 2, 0), (5, 3, 8), (1027, 2, 4)])
@pytest.mark.parametrize("below,above", [("s8", "s8"), ("s8", "f16"), ("f16", "s8"), ("u16", "u16")])
def test_any_format_over(ctx, below, above, w, h, pad):
    """'over' of two layers with padded rows and mixed formats into RGBA16F,
    with and without a colour matrix: within one f16 ulp of the FP64 result
    (1e-6 absolute near zero)."""
    tex = {"s8": (z.Texel(SB.UInt8x4, SP.RgbA), z.Color.SRGB), "f16": (z.Texel(SB.Float16x4, SP.RgbA), LINEAR),
           "u16": (z.Texel(SB.UInt16x4, SP.RgbA), z.Color.SRGB)}
    rng = np.random.default_rng([w, h, pad])

    def image(kind):
        t, c = tex[kind]
        pitch = w * t.bytes + pad if pad else 0
        d = z.Descriptor(w, h, t, c, pitch)
        if kind == "f16":
            raw = rng.random((h, w, 4)).astype(np.float16)
            return d, raw.view(np.uint8).reshape(h, -1), raw.astype(np.float64)
        dt, top = (np.uint8, 255.0) if kind == "s8" else (np.uint16, 65535.0)
        raw = rng.integers(0, int(top) + 1, (h, w, 4)).astype(dt)
        v = raw.astype(np.float64) / top
        v[..., :3] = C.eo_srgb(v[..., :3])
        return d, raw.view(np.uint8).reshape(h, -1), v

    (da, ra, va), (db, rb, vb) = image(below), image(above)
    lin = z.Texel(SB.Float16x4, SP.RgbA)
    for primaries in (z.Primaries.Bt709, z.Primaries.DisplayP3):
        cmd = z.CommandBuffer()
        a, b = cmd.input(da), cmd.input(db)
        # both layers in one declared chroma: linear f16 registers
        fa, fb = cmd.color_convert(a, LINEAR, lin), cmd.color_convert(b, LINEAR, lin)
        v = cmd.blend(fa, z.Rectangle(0, 0, w, h), fb)
        o, od = cmd.output(cmd.color_convert(v, z.Color(primaries=primaries, transfer=T.Linear), lin))
        out, exe = run_both(ctx, cmd, {a: da, b: db}, {a: ra, b: rb}, {o: od})
        # Tight images of in-line formats have a registered or compiled kernel.
        tag = "[any-format kernel]" if pad or below == "u16" else "[kernel "
        assert tag in exe.describe() and "interp" not in exe.describe()
        want = C.unpremultiply(C.over(C.premultiply(vb), C.premultiply(va)))
        if primaries != z.Primaries.Bt709:
            want[..., :3] = want[..., :3] @ C.convert_matrix(3, primaries, 5).T
        got = out[o].view(np.float16).reshape(h, w, 4)
        exp = C.encode_f16(want)
        ulp = np.abs(got.view(np.int16).astype(np.int32) - exp.view(np.int16).astype(np.int32))
        ulp = np.where(np.abs(got.astype(np.float64) - want) <= 1e-6, 0, ulp)
        visible = want[..., 3:] > 1e-3
        report(f"any_over_{below}_{above}", size=(w, h, pad), max_ulp=int(np.where(visible, ulp, 0).max()))
        assert np.where(visible, ulp, 0).max() <= 1
