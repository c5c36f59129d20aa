"""p2z_run_host from every mix of pageable and pinned buffers, at sizes around
its chunking (one block, one chunk, several chunks with a remainder, more
chunks than staging slots), in place, and with no layers: the words of the
device pass."""
from __future__ import annotations

import numpy as np
import pytest

import p2z

pytestmark = pytest.mark.gpu


def _device(ctx, trk, hit, nblocks, nl, W):
    dt, dh, do = ctx.upload(trk), ctx.upload(hit if hit.size else np.zeros(1, np.float32)), ctx.alloc(trk.nbytes)
    ctx.run(dt, dh, do, 1, nblocks, nl, W, "ref")
    out = ctx.download(do)
    for b in (dt, dh, do):
        b.free()
    return out


@pytest.mark.parametrize("W,nblocks,nl,nstreams", [(32, 1, 3, 0), (16, 7, 1, 0), (128, 5, 0, 0), (64, 601, 26, 0),
                                                   (128, 1111, 20, 1), (32, 6400, 20, 1), (32, 6403, 20, 2)])
def test_mixed_buffers(W, nblocks, nl, nstreams):
    rng = np.random.default_rng(nblocks)
    t, h, _, _ = p2z.generate("ref", 1, 4 * W, W, max(nl, 1))
    trk = np.tile(t.reshape(4, -1), (nblocks // 4 + 1, 1))[:nblocks].reshape(nblocks, 28, W).copy()
    trk[:, 4] += rng.normal(0, 1e-3, (nblocks, W)).astype(np.float32)
    trk = trk.reshape(-1)
    hit = np.tile(h.reshape(4, -1), (nblocks // 4 + 1, 1))[:nblocks].reshape(-1)[:nblocks * nl * 9 * W].copy()
    print(f"case host staging W={W} blocks={nblocks} layers={nl} slots={nstreams}", flush=True)
    with p2z.Context(0, nstreams=nstreams) as ctx:
        expect = _device(ctx, trk, hit, nblocks, nl, W).view(np.uint32)
        big = trk.nbytes + hit.nbytes > 50e6
        for mix in ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (1, 1, 1))[:2 if big else 6]:
            a = ctx.pinned_copy(trk) if mix[0] else trk.copy()
            b = (ctx.pinned_copy(hit) if mix[1] else hit.copy()) if hit.size else np.zeros(1, np.float32)
            out = ctx.pinned_empty(trk.size) if mix[2] else np.empty_like(trk)
            for _ in range(2):
                out[:] = 7.0
                ctx.run_host(a, b, out, 1, nblocks, nl, W, "ref")
                assert np.array_equal(out.view(np.uint32), expect), mix
            ctx.run_host(a, b, a, 1, nblocks, nl, W, "ref")
            assert np.array_equal(a.view(np.uint32), expect), ("in place", mix)
