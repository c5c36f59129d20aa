"""The report kernel (p2z_summary_device) at the edges of its work split:
fewer tracks than one workgroup's 2048, a remainder, events shorter than a
thread's stride, no accepted track, all widths; against exactly rounded sums
on the host.  A sum on the GPU is at most 64 additions deep at these sizes, so
a mean may be off by 64 * 2^-53 * mean|v|; an RMS is rounded to a float, so by
one float ulp."""
from __future__ import annotations

import math

import numpy as np
import pytest

import p2z

pytestmark = pytest.mark.gpu

LAST = np.array([15.5, 65.9, -189.5], np.float32)


def _tracks(rng, n):
    par = np.stack([LAST[0] * (1 + 0.2 * rng.normal(size=n)), LAST[1] * (1 + 0.1 * rng.normal(size=n)),
                    LAST[2] * (1 + 1e-6 * rng.normal(size=n)), 1 / (12.3 + rng.normal(size=n)),
                    1.3 + 0.2 * rng.normal(size=n), 2.8 + 0.1 * rng.normal(size=n)]).astype(np.float32)
    par[0, rng.random(n) < 0.02] = np.nan
    par[1, rng.random(n) < 0.02] = np.inf
    par[3, rng.random(n) < 0.02] = 0.0
    par[4, rng.random(n) < 0.02] = -0.1          # outside the window
    par[2, rng.random(n) < 0.02] = 2 * LAST[2]   # on its edge: accepted
    return par


def _expect(par):
    x = [p.astype(np.float64) for p in par]
    with np.errstate(divide="ignore"):
        x[3] = 1 / x[3]
    want = [float(v) for v in LAST] + [12.0, 1.3, 2.8]
    fin = np.all([np.isfinite(v) for v in x], axis=0)
    with np.errstate(invalid="ignore"):
        good = fin & np.all([~(np.abs((v - w) / w) > 1) for v, w in zip(x, want)], axis=0)
    x = [v[good] for v in x]
    vals = x[:3] + [(v - w) / v for v, w in zip(x[:3], want)] + x[3:]
    n = int(good.sum())
    counts = dict(nnans=int((~fin).sum()), nfail=int((fin & ~good).sum()), ngood=n)
    if n == 0:
        return [], [], [], counts
    means = [math.fsum(v) / n for v in vals]
    rms = [np.sqrt(np.float32(math.fsum((v - m) ** 2) / n)) for v, m in zip(vals[:6], means[:6])]
    return means, [math.fsum(np.abs(v)) / n for v in vals], rms, counts


@pytest.mark.parametrize("W,nevts,nb,ntrks", [(32, 1, 1, 1), (16, 1, 4, 63), (64, 1, 32, 2047), (64, 1, 32, 2048),
                                              (128, 3, 6, 683), (32, 1000, 1, 5), (16, 3, 200, 3199),
                                              (32, 7, 300, 9600)])
def test_summary_sizes(ctx, W, nevts, nb, ntrks):
    rng = np.random.default_rng(nevts * 31 + ntrks)
    blk = np.zeros((nevts, nb, 28, W), np.float32)
    blk[:, :, :6] = np.nan  # tracks past ntrks are not part of the report
    par = _tracks(rng, nevts * ntrks)
    for t in range(nevts * ntrks):
        ie, it = divmod(t, ntrks)
        blk[ie, it // W, :6, it % W] = par[:, t]
    print(f"case summary W={W} {nevts}x{ntrks}", flush=True)
    out = ctx.upload(blk.reshape(-1))
    try:
        for _ in range(2):
            s = ctx.summary_device(out, nevts, nb, W, ntrks, LAST).as_dict()
            means, scale, rms, counts = _expect(par)
            assert {k: s[k] for k in counts} == counts
            for k, m, a in zip(p2z.SUMMARY_FIELDS[:9], means, scale):
                assert abs(s[k] - m) <= 64 * 2.0 ** -53 * a, (k, s[k], m)
            for k, r in zip(p2z.SUMMARY_FIELDS[9:], rms):
                assert abs(s[k] - r) <= np.spacing(r), (k, s[k], r)
    finally:
        out.free()


def test_summary_without_an_accepted_track(ctx):
    blk = np.zeros(28 * 32 * 4, np.float32)
    out = ctx.upload(blk)
    s = ctx.summary_device(out, 1, 4, 32, 128, LAST).as_dict()
    out.free()
    assert (s["nnans"], s["nfail"], s["ngood"]) == (128, 0, 0)
    assert all(math.isnan(s[k]) for k in p2z.SUMMARY_FIELDS)
