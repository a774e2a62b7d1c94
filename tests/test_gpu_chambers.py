"""Sealed all-liquid chambers of one brick whose right-hand sides differ by many orders of magnitude: the coarse solve
makes each pure-Neumann component consistent by its own mean, at the component's own scale.

A wall of solid splits the grid.  One chamber moves fast; in the other all velocities are 0 and the volume correction
gives every cell the same right-hand side c.  The chamber has 256 unknowns, so its sum 256 c and its mean c are exact,
what is left of its right-hand side is 0, and its pressure stays exactly 0 however small c is beside the other chamber.
The bottom in one workgroup per grid (k_bottom) takes the same means as the separate launches, bit for bit.
"""
import os

import numpy as np
import pytest

import shiokaze_amd as S

pytestmark = pytest.mark.gpu


def chambers(w, h, d, wall, speed, seed=1):
    """Liquid everywhere, solid in the cells wall[0] <= i < wall[1]; velocities of `speed` before the wall, 0 behind it."""
    r = np.random.default_rng(seed)
    i = np.arange(w + 1)
    solid = np.broadcast_to(np.maximum(wall[0] - i, i - wall[1]) - 0.01, (d + 1, h + 1, w + 1)).T
    vel = []
    for shape in ((w + 1, h, d), (w, h + 1, d), (w, h, d + 1)):
        u = np.zeros(shape, np.float32)
        u[:wall[0] + 1] = speed * r.standard_normal((wall[0] + 1,) + shape[1:])
        vel.append(u)
    return S.Scene(w, h, d, 1.0 / 120.0, np.full((w, h, d), -1.0, np.float32), np.ascontiguousarray(solid, np.float32), *vel)


@pytest.mark.parametrize("precision", [S.PREC_FP64, S.PREC_MIXED])
@pytest.mark.parametrize("ratio", [1.0, 1e-6, 1e-12, 1e-16])
def test_each_chamber_by_its_own_mean(ratio, precision):
    print(f"[gpu-case] chambers ratio={ratio} precision={precision}", flush=True)
    speed = 1024.0
    # cells 0..1 fast, 2..3 solid, 4..7 at rest: 256 unknowns
    sc = chambers(8, 8, 8, (2, 4), speed)
    with S.Context(0) as ctx:
        excess = ratio * speed / 9.2  # the gain of the volume correction: about 9.2 per unit
        prm = S.default_params(residual=1e-2, precision=precision, current_volume=1.0 + excess, target_volume=1.0)
        r, _, P64 = ctx.project(sc, prm, pressure64=True)
    assert r.status == 0 and r.n_unknowns == 384 and r.n_levels == 1
    assert r.rhs_correct != 0.0
    assert np.abs(P64[:2]).max() > 0.0
    assert np.all(P64[4:] == 0.0), np.abs(P64[4:]).max()


@pytest.mark.parametrize("shape,wall", [((32, 16, 16), (15, 17)), ((16, 8, 8), (6, 10)), ((64, 17, 9), (40, 48))])
def test_bottom_takes_the_same_means(shape, wall):
    print(f"[gpu-case] chambers in the bottom {shape}", flush=True)
    sc = chambers(*shape, wall, 1.0)
    out = []
    for separate in (False, True):
        old = os.environ.pop("SHKZ_NO_BOTTOM", None)
        if separate:
            os.environ["SHKZ_NO_BOTTOM"] = "1"
        try:
            with S.Context(0) as ctx:
                work = sc.copy()
                prm = S.default_params(residual=1e-6, current_volume=1.0 + 1e-9, target_volume=1.0, max_iterations=40)
                r, _, P64 = ctx.project(work, prm, pressure64=True)
        finally:
            os.environ.pop("SHKZ_NO_BOTTOM", None)
            if old is not None:
                os.environ["SHKZ_NO_BOTTOM"] = old
        assert r.status == 0 and r.n_levels > 1
        out.append((r.iterations, P64))
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1].view(np.uint64), out[1][1].view(np.uint64))
