"""The bottom of the V-cycle in one workgroup per grid (k_bottom) against one launch per level and
step (SHKZ_NO_BOTTOM=1), and the oracle's own system: grids whose bottoms have one to four levels, odd
sides, long thin grids, 2D grids, pure-Neumann components, and several sweep counts.  Both forms give
the same bits."""
import os

import numpy as np
import pytest

import shiokaze_amd as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# name: (scene, w, h, d); d = 0 is a 2D grid
GRIDS = {
    "one_level": (S.SCENE_RANDOM_DROP, 16, 16, 16),
    "two_levels": (S.SCENE_RANDOM_DROP, 17, 25, 19),
    "odd_solids": (S.SCENE_DROP_SOLIDS, 41, 33, 47),
    "long_y": (S.SCENE_RANDOM_DROP, 9, 200, 8),
    "all_fluid": (S.SCENE_SMOKE, 20, 33, 17),
    "flat": (S.SCENE_DROP_SOLIDS, 90, 53, 0),
    "flat_thin": (S.SCENE_DROP, 7, 150, 0),
}
# (coarse sweeps per smoothing step, coarsest-brick sweeps)
CONTROLS = [(1, 48), (2, 1), (2, 7)]


def run(scene, flat, prm, separate):
    old = os.environ.pop("SHKZ_NO_BOTTOM", None)
    if separate:
        os.environ["SHKZ_NO_BOTTOM"] = "1"
    try:
        with S.Context(0) as ctx:
            work = scene.copy()
            r, _, P64 = (ctx.project2d if flat else ctx.project)(work, prm, pressure64=True)
    finally:
        os.environ.pop("SHKZ_NO_BOTTOM", None)
        if old is not None:
            os.environ["SHKZ_NO_BOTTOM"] = old
    assert r.status == 0 and r.converged, r.as_dict()
    return r, P64, work


@pytest.mark.parametrize("sweeps,coarsest", CONTROLS)
@pytest.mark.parametrize("name", list(GRIDS))
def test_bottom_in_one_workgroup(name, sweeps, coarsest):
    kind, w, h, d = GRIDS[name]
    print(f"[gpu-case] bottom {name} {w}x{h}x{d} sweeps {sweeps}/{coarsest}", flush=True)
    scene = S.make_scene2d(kind, w, h, seed=3) if d == 0 else S.make_scene(kind, w, h, d, seed=3)

    def prm(residual):
        return S.default_params(residual=residual, mg_coarse_pre_sweeps=sweeps, mg_coarse_post_sweeps=sweeps,
                                mg_coarse_sweeps=coarsest)

    # the same operations in the same order: the same bits, whatever the tolerance
    for residual in (1e-4, 1e-8):
        (one, P, a), (many, Q, b) = (run(scene, d == 0, prm(residual), separate) for separate in (False, True))
        assert one.iterations == many.iterations and one.reresid_inf == many.reresid_inf
        assert np.array_equal(P.view(np.uint64), Q.view(np.uint64))
        assert np.array_equal(a.u.view(np.uint32), b.u.view(np.uint32))
    if d:
        A = O.assemble(scene)
        x = O.gather(A, P)
        assert np.abs(A["b"] - O.spmv(A, x)).max() <= 1.01e-8 * np.abs(A["b"]).max()
