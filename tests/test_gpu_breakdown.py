"""A breakdown of the inner CG (p.q = 0: the residual's preconditioned image underflows) found by the kernels that form
their scalars themselves, against separate launches for the scalars (SHKZ_NO_FUSE=1): every workgroup stops before it
touches the iterate, so both report the same error with the same iterations and the same pressure.  Velocities near
FP32's smallest numbers, on grids from a few bricks to several hundred.
"""
import os

import numpy as np
import pytest

import shiokaze_amd as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def run(scene, separate):
    old = os.environ.pop("SHKZ_NO_FUSE", None)
    if separate:
        os.environ["SHKZ_NO_FUSE"] = "1"
    try:
        with S.Context(0) as ctx:
            work = scene.copy()
            r, _, P64 = ctx.project(work, S.default_params(residual=1e-6), pressure64=True, check=False)
    finally:
        os.environ.pop("SHKZ_NO_FUSE", None)
        if old is not None:
            os.environ["SHKZ_NO_FUSE"] = old
    return r, P64, work


@pytest.mark.parametrize("kind,side", [(S.SCENE_DROP, 16), (S.SCENE_RANDOM_DROP, 17), (S.SCENE_DROP_SOLIDS, 40),
                                       (S.SCENE_SPHERES_BOX, 64)])
def test_breakdown_leaves_the_iterate(kind, side):
    print(f"[gpu-case] breakdown {side}^3", flush=True)
    scene = S.make_scene(kind, side, seed=1)
    scale = 1e-41 / np.abs(O.assemble(scene)["b"]).max()
    for a in (scene.u, scene.v, scene.wv):
        a[...] = (a.astype(np.float64) * scale).astype(np.float32)
    (one, P, a), (many, Q, b) = (run(scene, separate) for separate in (False, True))
    assert one.status == many.status == S.ERR_NUMERIC
    assert one.iterations == many.iterations > 0
    assert np.all(np.isfinite(P)) and np.array_equal(P.view(np.uint64), Q.view(np.uint64))
    for x, y in ((a.u, b.u), (a.v, b.v), (a.wv, b.wv)):
        assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
