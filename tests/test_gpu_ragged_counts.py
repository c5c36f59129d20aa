"""The ragged passes' layer loop where lanes, blocks and waves end at different
layers: blocks without layers beside live ones in one wave, lanes shorter than
their block, a table that ends inside a wave; word for word against the
oracle's ragged driver, every launch form and hit-staging depth."""
from __future__ import annotations

import numpy as np
import pytest

import p2z
import pyoracle as O
from parity import random_blocks, same_words

pytestmark = pytest.mark.gpu

COUNTS = {"one": [1], "dead first": [0, 3, 0, 1, 2], "all dead": [0, 0, 0], "ends": [1, 2, 3, 4, 5, 6, 7],
          "long beside short": [9, 1, 1, 8, 2, 0, 0, 0, 5]}


@pytest.mark.parametrize("W", [16, 32, 64, 128])
@pytest.mark.parametrize("name", list(COUNTS))
def test_counts(ctx, W, name):
    counts = np.array(COUNTS[name], np.int32)
    nb, rng = len(counts), np.random.default_rng(W)
    blocks = [random_blocks(rng, W) for _ in range(nb)]
    trk = np.stack([b[0] for b in blocks]).reshape(nb, 28, W)
    hit = np.concatenate([np.repeat(blocks[b][1].reshape(1, 9, W), max(int(c), 0), 0) for b, c in enumerate(counts)]
                         + [np.zeros((1, 9, W), np.float32)])  # one record more, so that no array is empty
    first = np.concatenate([[0], np.cumsum(counts)[:-1]])
    for b, c in enumerate(counts):
        hit[first[b]:first[b] + c, 2] += (12.5 * np.arange(c, dtype=np.float32))[:, None]
    table = np.zeros(nb, p2z.BLOCK_DESC_DTYPE)
    table["trk_block"] = table["out_block"] = np.arange(nb)
    table["hit_block"], table["nlayer"] = first, counts
    lanes = np.repeat(counts, W) - (np.arange(nb * W) % 3).astype(np.int32)  # some lanes shorter, some below zero
    lanes = lanes.astype(np.int32)
    expect = O.run_ragged(trk.reshape(-1).copy(), hit.reshape(-1).copy(), nb, W, table["trk_block"].copy(),
                          table["hit_block"].copy(), table["nlayer"].copy(), np.maximum(lanes, 0))
    bufs = [ctx.upload(x) for x in (trk, hit, lanes, table.view(np.uint8))] + [ctx.alloc(trk.nbytes)]
    dt, dh, dl, db, do = bufs
    for opts in (dict(persistent=False, prefetch=1), dict(persistent=False, prefetch=2),
                 dict(waves_per_cu=1, prefetch=1), dict(waves_per_cu=1, prefetch=2)):
        ctx.h2d(do, np.zeros_like(trk))
        ctx.run_ragged(dt, dh, do, dl, db, nb, W, "ref", **opts)
        assert same_words(ctx.download(do), np.asarray(expect)), opts
    for b in bufs:
        b.free()
