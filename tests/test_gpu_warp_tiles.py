"""Tiles of the affine layer kernels whose taps all lie inside a layer's source
next to tiles that straddle its border: sources that hold the last tap of the
output exactly, by half a texel, or not, at whole and partial tiles."""
import numpy as np
import pytest

import zosimos_amd as z
from oracle import pipelines as PL
from zosimos_amd import workloads as W

from gpu_util import compare_u8, run

pytestmark = pytest.mark.gpu

SHIFTS = [(0.0, 0.0), (0.5, 0.5), (-0.5, -0.5), (-1.0, 0.0), (-130.25, -40.75), (96.0, 33.5)]


def _check(ctx, w, h, shift, few):
    """Two half-float layers, one as large as the output and one 200 x 60
    larger, shifted together: within 1 code of the FP64 oracle."""
    sizes = [(w, h), (w + 200, h + 60)]
    rng = np.random.default_rng([w, h])
    cmd = z.CommandBuffer()
    acc = cmd.solid_rgba(z.Descriptor.rgba16f_linear(w, h), (0.0, 0.0, 0.0, 0.0))
    aff = z.Affine.new(z.AffineSample.BiLinear).shift(*shift)
    inputs, host, layers = {}, {}, []
    for sw, sh in sizes:
        d = z.Descriptor.rgba16f_linear(sw, sh)
        r = cmd.input(d)
        acc = cmd.affine(acc, aff, r)
        inputs[r] = d
        host[r] = W.random_rgba16f(rng, sw, sh, rng.uniform(0.0, 1.0, (sh, sw)).astype(np.float32))
        layers.append(PL.f16_image(host[r], sw, sh))
    o, od = cmd.output(W.color_chain(cmd, acc))
    out, exe = run(ctx, cmd, inputs, host, {o: od})
    text = exe.describe()
    assert "[kernel w_" in text and ("kernel for few" in text) == few, text
    _, want = PL.c5(layers, [aff.transformation] * 2, (h, w))
    mr, ma, _ = compare_u8(f"warp_tiles_{w}x{h}_{shift[0]}_{shift[1]}", out[o], want, alpha_ok=want[..., 3] > 0)
    assert mr <= 1 and ma <= 1


# At most one tile per compute unit (256): every border test runs.
@pytest.mark.parametrize("shift", SHIFTS)
@pytest.mark.parametrize("w,h", [(64, 16), (256, 64), (301, 75)])
def test_border_tests_of_few_tiles(ctx, w, h, shift):
    _check(ctx, w, h, shift, True)


# 352 tiles: a grid resident as a whole, inside tiles without border tests.
@pytest.mark.parametrize("shift", SHIFTS)
def test_inside_and_border_tiles(ctx, shift):
    _check(ctx, 701, 512, shift, False)


# 2277 tiles, more than are resident (at most 2048: 8 workgroups of 4 waves a
# compute unit): dealt in runs of one tile, the last round of 8 x 64 of them
# partial.
@pytest.mark.parametrize("shift", [SHIFTS[1], SHIFTS[4]])
def test_runs_of_tiles(ctx, shift):
    _check(ctx, 2101, 1101, shift, False)


def test_longer_runs_of_tiles(ctx):
    """36,381 tiles: runs of two (at 5 resident workgroups a compute unit) and a
    last one of one tile, within 1 code of the interpreter where alpha is at
    least 8 codes."""
    w, h = 4281, 8681
    rng = np.random.default_rng(4)
    d = z.Descriptor.rgba16f_linear(w, h)
    cmd = z.CommandBuffer()
    r = cmd.input(d)
    canvas = cmd.solid_rgba(d, (0.0, 0.0, 0.0, 0.0))
    acc = cmd.affine(canvas, z.Affine.new(z.AffineSample.BiLinear).shift(-70.25, 20.5), r)
    o, od = cmd.output(W.color_chain(cmd, acc))
    block = W.random_rgba16f(rng, 977, 577, rng.uniform(0.0, 1.0, (577, 977)).astype(np.float32))
    tiled = np.tile(block.view(np.uint64).reshape(577, 977), (h // 577 + 1, w // 977 + 1))[:h, :w]
    host = {r: np.ascontiguousarray(tiled).view(np.uint8)}
    out, exe = run(ctx, cmd, {r: d}, host, {o: od})
    assert "[kernel w_h_chain_s8" in exe.describe()
    ref, _ = run(ctx, cmd, {r: d}, host, {o: od}, flags=z.PLAN_INTERPRETER)
    got, want = (x[o].reshape(h, w, 4) for x in (out, ref))
    diff = np.maximum(got, want) - np.minimum(got, want)
    assert diff[..., 3].max() <= 1 and diff[want[..., 3] >= 8].max() <= 1
