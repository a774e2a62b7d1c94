"""NaN samples in the level set: a liquid cell beside one keeps its couplings but has no diagonal, so that its pressure
stays 0.  The prolongation inside the first post-smoothing application must leave such cells alone on every level, across
the faces of its brick too: the same iterations and bits as a launch of its own (SHKZ_NO_JOIN=1).  Single samples, and
blocks whose shell of such cells fills whole cells of the coarser levels."""
import os

import numpy as np
import pytest

import shiokaze_amd as S

pytestmark = pytest.mark.gpu


def run(scene, flat, prm, separate):
    old = os.environ.pop("SHKZ_NO_JOIN", None)
    if separate:
        os.environ["SHKZ_NO_JOIN"] = "1"
    try:
        with S.Context(0) as ctx:
            work = scene.copy()
            r, _, P64 = (ctx.project2d if flat else ctx.project)(work, prm, pressure64=True)
    finally:
        os.environ.pop("SHKZ_NO_JOIN", None)
        if old is not None:
            os.environ["SHKZ_NO_JOIN"] = old
    assert r.status == 0 and r.converged
    return r, P64


@pytest.mark.parametrize("edge", [1, 2, 3, 5])
@pytest.mark.parametrize("shape", [(37, 30, 29), (64, 40, 48), (60, 45), (170, 90)])
def test_joined_prolongation_beside_nan(shape, edge):
    print(f"[gpu-case] NaN blocks of {edge} in {shape}", flush=True)
    flat = len(shape) == 2
    scene = (S.make_scene2d if flat else S.make_scene)(S.SCENE_DROP_SOLIDS, *shape, seed=1)
    rng = np.random.default_rng(edge)
    for _ in range(30):
        at = [int(rng.integers(0, n - edge)) for n in shape]
        scene.fluid[tuple(slice(a, a + edge) for a in at)] = np.nan
    prm = S.default_params(residual=1e-6)
    (one, P), (two, Q) = (run(scene, flat, prm, separate) for separate in (False, True))
    assert np.all(np.isfinite(P))
    assert one.iterations == two.iterations
    assert np.array_equal(P.view(np.uint64), Q.view(np.uint64))
