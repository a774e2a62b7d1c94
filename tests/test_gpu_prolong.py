"""The prolongation joined to the first post-smoothing, where its tile can go wrong: bricks at odd and even places
of their coarse brick along each axis, coarse rows in missing bricks, ragged ends, one layer (2D), with every
number of smoothing steps that it can precede.  The solve to 1e-9 must meet its residual in FP64 against
the oracle's operator.
"""
import numpy as np
import pytest

import shiokaze_amd as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(17, 33, 9), (25, 16, 41), (64, 17, 31), (40, 72, 24), (9, 90, 15)]
SHAPES_2D = [(33, 150), (96, 71)]


@pytest.fixture(scope="module")
def ctx():
    c = S.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("post", [1, 2])
@pytest.mark.parametrize("local", [2, 3])
@pytest.mark.parametrize("shape", SHAPES + SHAPES_2D)
def test_vcycle_with_joined_prolongation(ctx, shape, local, post):
    print(f"[gpu-case] prolongation {shape} local={local} post={post}", flush=True)
    flat = len(shape) == 2
    sc = (S.make_scene2d if flat else S.make_scene)(S.SCENE_DROP_SOLIDS, *shape, seed=sum(shape))
    A = (O.assemble2 if flat else O.assemble)(sc)
    prm = S.default_params(residual=1e-9, precision=S.PREC_MIXED, mg_smoother=S.SMOOTH_BRICK, mg_local_sweeps=local,
                           mg_pre_sweeps=post, mg_post_sweeps=post, mg_coarse_pre_sweeps=post, mg_coarse_post_sweeps=post)
    r, P, P64 = (ctx.project2d if flat else ctx.project)(sc, prm, pressure64=True)
    assert r.status == 0 and r.converged
    resid = A["b"] - O.spmv(A, O.gather(A, P64))
    assert np.abs(resid).max() <= 1e-9 * np.abs(A["b"]).max() * 1.0001
