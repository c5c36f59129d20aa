"""The work queue where its counters hand out items (a grid with fewer waves than
items, so that most chunks come from the counters): every arithmetic, width,
hit-staging depth and claim, eager and captured, with blocks without layers, at
full size, from several threads, and under the batching server.  Reference
typing word for word against the oracle; the others against the launch of one
wave per item, whose accuracy tests/test_gpu_precision.py measures."""
from __future__ import annotations

import threading

import numpy as np
import pytest

import p2z
import pyoracle as O
from parity import same_words
from test_gpu_ragged import SMALL_GRID, Dev, oracle_ragged
from test_gpu_serve import event_blocks

pytestmark = pytest.mark.gpu

WAVES = 256  # of SMALL_GRID: one per CU of 256


def _items(w, blocks=None):
    return ((w.nblocks if blocks is None else blocks) * w.width + 63) // 64


@pytest.fixture(scope="module", params=[16, 32, 64, 128])
def table(ctx, request):
    w = p2z.Workload("ragged", nevents=40, width=request.param, seed=6)
    d = Dev(ctx, w)
    yield w, d, oracle_ragged(w)
    d.free()
    w.close()


@pytest.mark.parametrize("prefetch", [1, 2])
@pytest.mark.parametrize("claim,graph", [(1, False), (1, True), (3, False)])
def test_reference_typing_past_the_first_chunks(ctx, table, claim, graph, prefetch):
    w, d, expect = table
    assert _items(w) > 2 * WAVES * claim
    for rep in range(3):
        ctx.h2d(d.out, np.zeros(w.tracks.size, np.float32))
        ctx.run_ragged(d.trk, d.hit, d.out, d.lanes, d.blk, w.nblocks, w.width, "ref", graph=graph,
                       **dict(SMALL_GRID, items_per_claim=claim, prefetch=prefetch))
        assert same_words(ctx.download(d.out), expect), rep


def test_blocks_without_layers(ctx, table):
    w, d, _ = table
    blocks = np.array(w.blocks, copy=True)
    blocks["nlayer"][::7] = 0
    blocks["nlayer"][3::5] = np.minimum(blocks["nlayer"][3::5], 1)
    expect = O.run_ragged(w.tracks, w.hits, w.nblocks, w.width, blocks["trk_block"], blocks["hit_block"],
                          blocks["nlayer"], w.lane_nlayer)
    dblk = ctx.upload(np.ascontiguousarray(blocks))
    ctx.h2d(d.out, np.zeros(w.tracks.size, np.float32))
    ctx.run_ragged(d.trk, d.hit, d.out, d.lanes, dblk, w.nblocks, w.width, "ref", **SMALL_GRID)
    got = ctx.download(d.out)
    dblk.free()
    assert same_words(got, expect)


def test_full_size(ctx):
    """2000 events, 6.3e6 tracks: reference typing against the oracle, FAST and
    the FP64 gain steps against one wave per item."""
    w = p2z.Workload("ragged", nevents=2000, width=32, seed=2024)
    d = Dev(ctx, w)
    shape = dict(tracks_per_wg=256, prefetch=1, waves_per_cu=8, items_per_claim=2)

    def run(math, **opts):
        ctx.h2d(d.out, np.zeros(w.tracks.size, np.float32))
        ctx.run_ragged(d.trk, d.hit, d.out, d.lanes, d.blk, w.nblocks, 32, math, **opts)
        return ctx.download(d.out)

    assert _items(w) > 8 * WAVES * 2
    for math in ("fast", "fp64gain"):
        print(f"case queue/full-size {math}", flush=True)
        assert same_words(run(math, graph=True, **shape), run(math, persistent=False)), math
    print("case queue/full-size ref", flush=True)
    assert same_words(run("ref", graph=True, **shape), oracle_ragged(w))
    d.free()
    w.close()


def test_contexts_on_threads():
    """Each context's queue counters are its own."""
    w = p2z.Workload("ragged", nevents=40, width=32, seed=7)
    expect = oracle_ragged(w)
    start, differ, failures = threading.Barrier(4), [], []

    def work(k):
        try:
            with p2z.Context(0) as c:
                d = Dev(c, w)
                start.wait(timeout=60)
                for rep in range(10):
                    c.run_ragged(d.trk, d.hit, d.out, d.lanes, d.blk, w.nblocks, 32, "ref", graph=rep % 2 == 1,
                                 **SMALL_GRID)
                    if not same_words(c.download(d.out), expect):
                        differ.append((k, rep))
                d.free()
        except Exception as e:  # reported below, in the main thread
            failures.append(repr(e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not any(t.is_alive() for t in threads), "a thread did not finish"
    assert not failures and not differ, (failures, differ)
    w.close()


@pytest.mark.parametrize("math", ["ref", "fp64gain"])
@pytest.mark.parametrize("opts", [SMALL_GRID, dict(items_per_claim=2), dict(waves_per_cu=1, prefetch=2)])
def test_batching_server(ctx, math, opts):
    """Batches on the queue, several in flight, each batch's items more than its
    grid's waves or claims."""
    w = p2z.Workload("ragged", nevents=60, width=32, seed=8)
    d = Dev(ctx, w, lpt=False)
    if math == "ref":
        expect = oracle_ragged(w)
    else:
        ctx.run_ragged(d.trk, d.hit, d.out, d.lanes, d.blk, w.nblocks, 32, math, persistent=False)
        expect = ctx.download(d.out)
    with p2z.Server(ctx, d.trk, d.hit, d.lanes, 2 * w.tracks.nbytes, 32, math, nstreams=2, **opts) as sv:
        for rnd in range(2):
            ids = list(range(rnd * 1000, rnd * 1000 + w.nevents))
            for r in ids:
                assert sv.submit(r, event_blocks(w, r % 1000)) == p2z.OK
            done = sv.wait(ids)
            for r in ids:
                b0, b1 = int(w.event_blocks[r % 1000]), int(w.event_blocks[r % 1000 + 1])
                assert same_words(sv.result(done[r]), expect[b0 * 28 * 32:b1 * 28 * 32]), (rnd, r)
                sv.release(r)
    d.free()
    w.close()
