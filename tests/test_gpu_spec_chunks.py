"""The chunks of a pointwise batch: images that end just below, at and just
above a chunk of one or of two steps (1024 pixels a step)."""
import numpy as np
import pytest

import zosimos_amd as z
from oracle import pipelines as PL
from zosimos_amd import workloads as W

from gpu_util import compare_u8, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("large", [None, (2049, 2049)])
def test_chunk_edges(ctx, large):
    """Without a large image chunks are of one step; with 4.2 million pixels
    on 256 compute units of two.  Within 1 code of the FP64 oracle."""
    sizes = [(1023, 1), (1024, 1), (1025, 1), (2047, 1), (2048, 1), (2049, 1), (1, 3), (64, 64)]
    sizes += [large] if large else []
    cmd = z.CommandBuffer()
    ins, outs, host, regs = {}, {}, {}, []
    rng = np.random.default_rng(9)
    for w, h in sizes:
        d = z.Descriptor.rgba8_srgb(w, h)
        r = cmd.input(d)
        o, od = cmd.output(W.color_chain(cmd, r))
        ins[r], outs[o] = d, od
        host[r] = rng.integers(0, 256, (h, w * 4), dtype=np.uint8)
        regs.append((r, o, w, h))
    out, exe = run(ctx, cmd, ins, host, outs)
    assert exe.stats()[0] == 1
    for r, o, w, h in regs:
        _, want = PL.c4(PL.u8_image(host[r], w, h))
        mr, ma, _ = compare_u8(f"chunk_edges_{w}x{h}", out[o], want)
        assert mr <= 1 and ma == 0
