"""What a track that is outside the reference typing's short layer step costs its
wave (p2z-tests_amd/csrc/p2z_lane.hpp): where it is from the first layer on, the
full steps alone; where it is later, the short steps and then the full ones.
Every wave alone on its SIMD, so that the time of the pass is the time of its
slowest wave; a full layer step is below 1.5 short ones (671 against 460
instructions)."""
from __future__ import annotations

import numpy as np
import pytest

import p2z

pytestmark = pytest.mark.gpu

W, NL, NB = 32, 20, 256  # 128 waves


def _unused_lane(trk, hit):
    """The last lane of every block left at zero, as in a partly used block."""
    trk[:, :, W - 1] = 0.0
    hit[:, :, :, W - 1] = 0.0


def _not_finite(trk, hit):
    trk[:, 0, 3] = np.nan


def _layer_at_z_zero(trk, hit):
    hit[:, 2, 2] = 0.0


def _hit_z_missing(trk, hit):
    hit[:, 2, 2, 7] = np.nan


@pytest.mark.parametrize("change,most", [(_unused_lane, 1.7), (_not_finite, 1.7), (_layer_at_z_zero, 1.2),
                                         (_hit_z_missing, 2.7)])
def test_cost_of_a_wave_with_a_track_outside(ctx, change, most):
    trk, hit, _, nb = p2z.generate("ref", 1, NB * W, W, NL)
    t, h = trk.reshape(nb, 28, W).copy(), hit.reshape(nb, NL, 9, W).copy()
    change(t, h)
    print(f"case cost of {change.__name__}", flush=True)
    dt, dh, do = ctx.upload(trk), ctx.upload(hit), ctx.alloc(trk.nbytes)
    bt, bh = ctx.upload(t.reshape(-1)), ctx.upload(h.reshape(-1))

    def us(a, b):
        best = []
        for _ in range(30):
            ctx.timer_start()
            for _ in range(20):
                ctx.run(a, b, do, 1, nb, NL, W, "ref")
            best.append(ctx.timer_stop() / 20 * 1e3)
        return min(best)

    plain, with_it = us(dt, dh), us(bt, bh)
    for b in (dt, dh, do, bt, bh):
        b.free()
    print(f"  plain {plain:.1f} us, with it {with_it:.1f} us: {with_it / plain:.2f}", flush=True)
    assert with_it <= most * plain
