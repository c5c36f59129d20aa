"""The reference typing's short layer step against the oracle, word for word,
where its conditions fail: operands outside its ranges, zeros of either sign,
values that are not finite (propagate_ref in p2z-tests_amd/csrc/p2z_lane.hpp).
NaN results compare equal to NaN (their sign and payload differ between CPUs
and GPUs)."""
from __future__ import annotations

import numpy as np
import pytest

import p2z
import pyoracle as O
from parity import random_blocks

pytestmark = pytest.mark.gpu

W, NB, NL = 32, 8, 5
PHI, THETA, IPT = 4, 5, 3
INF = np.float32(np.inf)


def _set_hit(word, value):
    return lambda trk, hit, b, l, lay: hit.__setitem__((b, lay, word, l), value)


def _set_trk(word, value):
    return lambda trk, hit, b, l, lay: trk.__setitem__((b, word, l), value)


SPECIAL = {
    "plain": lambda *a: None,
    "z is +0": _set_hit(2, np.float32(0.0)),
    "z is -0": _set_hit(2, np.float32(-0.0)),
    "z far": _set_hit(2, np.float32(3e9)),
    "z infinite": _set_hit(2, INF),
    "z NaN": _set_hit(2, np.float32(np.nan)),
    "hit x infinite": _set_hit(0, -INF),
    "hit x NaN": _set_hit(0, np.float32(np.nan)),
    "hit cov infinite": _set_hit(3, INF),
    "hit cov huge": _set_hit(5, np.float32(1e30)),
    "phi large": _set_trk(PHI, np.float32(500.25)),
    "phi at 120": _set_trk(PHI, np.float32(120.0)),
    "theta large": _set_trk(THETA, np.float32(-1234.5)),
    "theta next to pi/2": _set_trk(THETA, np.float32(np.pi / 2)),
    "turn above 0.75": _set_trk(THETA, np.float32(1.53)),
    "ipt zero": _set_trk(IPT, np.float32(0.0)),
    "ipt tiny": _set_trk(IPT, np.float32(1e-38)),
    "ipt subnormal": _set_trk(IPT, np.float32(1e-40)),
    "ipt huge": _set_trk(IPT, np.float32(2e9)),
    "charge zero": lambda trk, hit, b, l, lay: trk.view(np.int32).__setitem__((b, 27, l), 0),
    "cov -0": _set_trk(6 + 13, np.float32(-0.0)),
    "cov all +0": lambda trk, hit, b, l, lay: trk.__setitem__((b, slice(6, 27), l), np.float32(0.0)),
    "cov all -0": lambda trk, hit, b, l, lay: trk.__setitem__((b, slice(6, 27), l), np.float32(-0.0)),
    "cov infinite": _set_trk(6 + 9, INF),
}


def _inputs(change):
    rng = np.random.default_rng(11)
    blocks = [random_blocks(rng, W) for _ in range(NB)]
    trk = np.stack([b[0] for b in blocks]).reshape(NB, 28, W)
    hit = np.empty((NB, NL, 9, W), np.float32)
    for b in range(NB):
        for lay in range(NL):
            hit[b, lay] = blocks[b][1].reshape(9, W)
            hit[b, lay, 2] += np.float32(12.5 * lay)
    # one lane of each half block, at every layer in turn, and a whole block
    for b in range(NB - 1):
        change(trk, hit, b, (5 * b) % 16, b % NL)
        change(trk, hit, b, 16 + (3 * b) % 16, (b + 2) % NL)
    for l in range(W):
        change(trk, hit, NB - 1, l, 3)
    return trk.reshape(-1).copy(), hit.reshape(-1).copy()


def _same(a, b):
    nan = np.isnan(a) & np.isnan(b)
    return bool(np.all((a.view(np.uint32) == b.view(np.uint32)) | nan))


@pytest.mark.parametrize("name", list(SPECIAL))
def test_operands_outside_the_short_form(ctx, name):
    with np.errstate(all="ignore"):
        trk, hit = _inputs(SPECIAL[name])
    print(f"case {name}", flush=True)
    for nl in (1, 2, NL):
        h = np.ascontiguousarray(hit.reshape(NB, NL, -1)[:, :nl]).reshape(-1)
        expect = O.run(trk, h, 1, NB, W, nl)
        dt, dh, do = ctx.upload(trk), ctx.upload(h), ctx.alloc(trk.nbytes)
        ctx.run(dt, dh, do, 1, NB, nl, W, "ref")
        got = ctx.download(do)
        ctx.run(dt, dh, dt, 1, NB, nl, W, "ref")  # in place
        again = ctx.download(dt)
        # the same tracks as a descriptor table, in both launch forms
        table = np.zeros(NB, p2z.BLOCK_DESC_DTYPE)
        table["trk_block"] = table["out_block"] = np.arange(NB)
        table["hit_block"], table["nlayer"] = np.arange(NB) * nl, nl
        dl, db = ctx.upload(np.full(NB * W, nl, np.int32)), ctx.upload(table.view(np.uint8))
        ctx.h2d(dt, trk)
        for persistent in (True, False):
            ctx.run_ragged(dt, dh, do, dl, db, NB, W, "ref", persistent=persistent, waves_per_cu=1)
            assert np.array_equal(ctx.download(do).view(np.uint32), got.view(np.uint32)), persistent
        for b in (dt, dh, do, dl, db):
            b.free()
        bad = np.flatnonzero((got.view(np.uint32) != expect.view(np.uint32)) & ~(np.isnan(got) & np.isnan(expect)))
        assert _same(got, expect), (nl, [(int(i) // (28 * W), int(i) // W % 28, int(i) % W) for i in bad[:5]],
                                    got[bad[:5]], expect[bad[:5]])
        assert np.array_equal(again.view(np.uint32), got.view(np.uint32))
