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


@pytest.mark.parametrize("shift", [(0.0, 0.0), (0.5, 0.5), (-0.5, -0.5), (-1.0, 0.0), (-130.25, -40.75), (96.0, 33.5)])
@pytest.mark.parametrize("w,h", [(64, 16), (256, 64), (301, 75)])
def test_inside_and_border_tiles(ctx, w, h, shift):
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
    assert "[kernel" in exe.describe()
    _, want = PL.c5(layers, [aff.transformation] * 2, (h, w))
    mr, ma, _ = compare_u8(f"warp_tiles_{w}x{h}_{shift[0]}_{shift[1]}", out[o], want, alpha_ok=want[..., 3] > 0)
    assert mr <= 1 and ma <= 1
