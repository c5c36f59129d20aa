"""The fused pass with the library's own hit-staging depth on both sides of the
size where the depth changes (16 waves per CU, default_hit_stage in
p2z-tests_amd/csrc/p2z_internal.hpp), against the depths set by the caller.  The
depth decides when a hit is loaded, not what is computed with it: every word is
equal."""
from __future__ import annotations

import numpy as np
import pytest

import p2z
from parity import random_blocks

pytestmark = pytest.mark.gpu

EDGE = 16 * 256 * 64  # tracks of 16 waves on each of 256 CUs


@pytest.mark.parametrize("W,ntracks,nlayer", [(16, 16, 1), (32, 96, 2), (64, EDGE, 3), (128, EDGE + 128, 4)])
@pytest.mark.parametrize("math", ["fast", "ref", "fp64gain"])
def test_depths_agree(ctx, W, ntracks, nlayer, math):
    rng = np.random.default_rng(W)
    nb, pool = ntracks // W, [random_blocks(rng, W) for _ in range(8)]
    trk = np.stack([pool[b % 8][0].reshape(28, W) for b in range(nb)])
    hit = np.stack([[pool[b % 8][1].reshape(9, W)] * nlayer for b in range(nb)])
    hit[:, :, 2] += (12.5 * np.arange(nlayer, dtype=np.float32))[None, :, None]
    dt, dh, do = ctx.upload(trk), ctx.upload(hit), ctx.alloc(trk.nbytes)
    outs = []
    try:
        for depth in (0, 1, 2):
            ctx.set_opts(hit_stage=depth)
            ctx.run(dt, dh, do, 1, nb, nlayer, W, math)
            outs.append(ctx.download(do).view(np.uint32))
    finally:
        ctx.set_opts()
        for b in (dt, dh, do):
            b.free()
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
