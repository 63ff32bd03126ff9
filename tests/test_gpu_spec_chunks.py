"""The chunks of a pointwise batch: images that end just below, at and just
above a chunk of 1, 2, 3 or 16 steps (1024 pixels a step), on the registered
batch kernel and on one compiled at run time."""
import numpy as np
import pytest

import zosimos_amd as z
from oracle import color as C
from oracle import pipelines as PL
from zosimos_amd import workloads as W

from gpu_util import compare_u8, run

pytestmark = pytest.mark.gpu

# Registered: sRGB texels; compiled: linear ones, a signature of no registered
# kernel.
TRANSFER = {"registered": z.Transfer.Srgb, "compiled": z.Transfer.Linear}


def _program(kind, sizes):
    """Independent images of one signature; [(input, output, w, h)]."""
    cmd, ins, outs, regs = z.CommandBuffer(), {}, {}, []
    for w, h in sizes:
        d = z.Descriptor(w, h, W.RGBA8, z.Color(transfer=TRANSFER[kind]))
        r = cmd.input(d)
        o, od = cmd.output(W.color_chain(cmd, r))
        ins[r], outs[o] = d, od
        regs.append((r, o, w, h))
    return cmd, ins, outs, regs


# With a large image chunks are of as many steps as leave 8 to each of 256
# compute units, 16 at most: 2.1 million pixels a step.
@pytest.mark.parametrize("steps,large", [(1, None), (2, (2049, 2049)), (3, (3001, 2200)), (16, (6401, 5600))])
@pytest.mark.parametrize("kind", list(TRANSFER))
def test_chunk_edges(ctx, kind, steps, large):
    """Each image within 1 code of the FP64 oracle, the large one equal to its
    own launch alone (a persistent grid, no chunks)."""
    chunk = 1024 * steps
    sizes = [(1023, 1), (1024, 1), (1025, 1), (2047, 1), (2048, 1), (2049, 1), (1, 3), (64, 64)]
    sizes += [(n, 1) for c in (chunk, 2 * chunk) for n in (c - 1, c, c + 1, c + 5)]
    sizes += [large] if large else []
    cmd, ins, outs, regs = _program(kind, sizes)
    rng = np.random.default_rng(9)
    host = {r: rng.integers(0, 256, (h, w * 4), dtype=np.uint8) for r, _, w, h in regs}
    out, exe = run(ctx, cmd, ins, host, outs)
    text = exe.describe()
    assert exe.stats()[0] == 1 and ("[kernel jit#" in text) == (kind == "compiled") and "unavailable" not in text
    for r, o, w, h in regs:
        if (w, h) == large:
            alone = _program(kind, [large])
            (r1, o1, _, _), = alone[3]
            ref, _ = run(ctx, *alone[:2], {r1: host[r]}, alone[2])
            assert np.array_equal(out[o], ref[o1])
            continue
        want = C.encode_u8(PL.chain(C.decode_u8(PL.u8_image(host[r], w, h), TRANSFER[kind])), 5)
        mr, ma, _ = compare_u8(f"chunk_edges_{kind}_{steps}_{w}x{h}", out[o], want)
        assert mr <= 1 and ma == 0
