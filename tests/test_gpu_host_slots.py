"""p2z_run_host where staging slots are used again: more chunks than slots, from
every mix of pageable and pinned track, hit and output buffers, each block with
tracks and hits of its own, so that a slot refilled, computed or emptied too
early changes the result.  Chunks are at least 32 MB, so the inputs are larger
than that for every slot."""
from __future__ import annotations

import itertools

import numpy as np
import pytest

import p2z

pytestmark = pytest.mark.gpu

W, NL, CHUNK = 32, 20, 32 << 20
BLOCK = (28 + 9 * NL) * W * 4


@pytest.fixture(scope="module")
def inputs():
    nblocks = 2 * 5 * CHUNK // BLOCK + 7  # 5 chunks for each of two slots, and a remainder
    t, h, _, _ = p2z.generate("ref", 1, 8 * W, W, NL)
    rng = np.random.default_rng(12)
    trk = np.tile(t.reshape(8, 28, W), (nblocks // 8 + 1, 1, 1))[:nblocks].copy()
    hit = np.tile(h.reshape(8, NL, 9, W), (nblocks // 8 + 1, 1, 1, 1))[:nblocks].copy()
    trk[:, 4] += rng.normal(0, 1e-3, (nblocks, W)).astype(np.float32)
    hit[:, :, 0] += rng.normal(0, 1e-3, (nblocks, 1, W)).astype(np.float32)
    return nblocks, trk.reshape(nblocks, -1), hit.reshape(nblocks, -1)


@pytest.mark.parametrize("nstreams", [1, 2])
@pytest.mark.parametrize("mix", list(itertools.product((0, 1), repeat=3)))
def test_slots_used_again(ctx, inputs, mix, nstreams):
    nblocks, trk, hit = inputs
    nblocks = nblocks if nstreams == 2 else nblocks // 2
    assert nblocks * BLOCK > 4 * nstreams * CHUNK
    trk, hit = trk[:nblocks].reshape(-1), hit[:nblocks].reshape(-1)
    dt, dh, do = ctx.upload(trk), ctx.upload(hit), ctx.alloc(trk.nbytes)
    ctx.run(dt, dh, do, 1, nblocks, NL, W, "ref")
    expect = ctx.download(do).view(np.uint32)
    for b in (dt, dh, do):
        b.free()
    print(f"case slots={nstreams} pinned={mix}", flush=True)
    with p2z.Context(0, nstreams=nstreams) as c:
        a = c.pinned_copy(trk) if mix[0] else trk
        b = c.pinned_copy(hit) if mix[1] else hit
        out = c.pinned_empty(trk.size) if mix[2] else np.empty_like(trk)
        for rep in range(2):
            out[:] = 7.0
            c.run_host(a, b, out, 1, nblocks, NL, W, "ref")
            assert np.array_equal(out.view(np.uint32), expect), rep
