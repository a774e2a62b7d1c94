"""The prolongation inside the first post-smoothing application (k_post_local4<.., PRO=1>) against a launch of its own
(k_prolong4, SHKZ_NO_JOIN=1) followed by the same smoothing: the same operations in the same order, so the same
iterations and the same bits.  Bricks at odd and even places of their coarse brick along each axis, coarse rows in
missing bricks, ragged ends, one layer (2D), bricks with a constant operator, the last application with and without the
partials of r.z, a batch whose grids end on different levels.
"""
import os

import numpy as np
import pytest

import shiokaze_amd as S

pytestmark = pytest.mark.gpu

SHAPES = [(17, 33, 9), (25, 16, 41), (64, 17, 31), (40, 72, 24), (9, 90, 15), (72, 88, 56)]
SHAPES_2D = [(33, 150), (96, 71), (260, 140)]


def bits(a):
    return a.view(np.uint64 if a.dtype == np.float64 else np.uint32)


def run(scenes, flat, prm, separate, bottom):
    env = {"SHKZ_NO_JOIN": separate, "SHKZ_NO_BOTTOM": not bottom}
    old = {k: os.environ.pop(k, None) for k in env}
    os.environ.update({k: "1" for k, on in env.items() if on})
    try:
        with S.Context(0) as ctx:
            work = [s.copy() for s in scenes]
            if len(work) > 1:
                res, _, P = ctx.project_batch(work, prm, pressure64=True)
            else:
                r, _, p = (ctx.project2d if flat else ctx.project)(work[0], prm, pressure64=True)
                res, P = [r], [p]
    finally:
        for k, v in old.items():
            os.environ.pop(k, None)
            if v is not None:
                os.environ[k] = v
    for r in res:
        assert r.status == 0 and r.converged
    return [r.iterations for r in res], list(P) + [w.u for w in work]


def same(scenes, flat, prm, bottom=True):
    (one, a), (two, b) = (run(scenes, flat, prm, separate, bottom) for separate in (False, True))
    assert one == two
    for x, y in zip(a, b):
        assert np.array_equal(bits(x), bits(y))


@pytest.mark.parametrize("post", [1, 2])
@pytest.mark.parametrize("local", [2, 3])
@pytest.mark.parametrize("shape", SHAPES + SHAPES_2D)
def test_joined_prolongation_keeps_the_bits(shape, local, post):
    print(f"[gpu-case] prolongation forms {shape} local={local} post={post}", flush=True)
    flat = len(shape) == 2
    scene = (S.make_scene2d if flat else S.make_scene)(S.SCENE_DROP_SOLIDS, *shape, seed=sum(shape))
    prm = S.default_params(residual=1e-9, precision=S.PREC_MIXED, mg_smoother=S.SMOOTH_BRICK, mg_local_sweeps=local,
                           mg_pre_sweeps=post, mg_post_sweeps=post, mg_coarse_pre_sweeps=post, mg_coarse_post_sweeps=post)
    same([scene], flat, prm)


@pytest.mark.parametrize("kind,shape", [(S.SCENE_SMOKE, (56, 40, 72)), (S.SCENE_SPHERES_BOX, (66, 50, 35))])
def test_every_level_joined(kind, shape):
    """Uniform bricks (an all-liquid grid), and every coarse level through the joined kernel."""
    print(f"[gpu-case] prolongation forms {shape}, no bottom", flush=True)
    same([S.make_scene(kind, *shape, seed=2)], False, S.default_params(residual=1e-6), bottom=False)


def test_batch_of_different_depths():
    print("[gpu-case] prolongation forms, batch", flush=True)
    scenes = [S.make_scene(S.SCENE_RANDOM_DROP, n, seed=n) for n in (8, 17, 40, 72)]
    same(scenes, False, S.default_params(residual=1e-6))
