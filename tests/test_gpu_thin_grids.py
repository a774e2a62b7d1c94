"""Long grids of few cells per plane, whose output takes several slabs of planes per workgroup (k_output<1>, up to 128
cells a plane): around that limit, with lengths that leave the last workgroup and the last slab partly empty, against
the oracle bit for bit; and a batch that holds both kinds, each grid as when projected alone.  Without any liquid, too.
"""
import numpy as np
import pytest

import shiokaze_amd as S
import test_gpu_grids as grids
from oracle import oracle as O

pytestmark = pytest.mark.gpu

ctx = grids.ctx
SHAPES = [(301, 2, 2), (1023, 1, 1), (250, 5, 7), (37, 16, 8), (130, 1, 127), (66, 128, 1), (38, 43, 3), (75, 13, 11)]
SHAPES_2D = [(1021, 1), (150, 2), (301, 37), (33, 127), (77, 128), (78, 129)]


@pytest.mark.parametrize("solid", [False, True])
@pytest.mark.parametrize("shape", SHAPES + SHAPES_2D)
def test_thin_grids_match_oracle(ctx, shape, solid):
    grids.test_grid_kernels_match_oracle(ctx, shape, solid)


def test_batch_of_thin_and_thick_grids(ctx):
    print("[gpu-case] thin and thick grids", flush=True)
    shapes = [(301, 2, 2), (20, 20, 20), (37, 16, 8), (9, 30, 41), (1023, 1, 1), (66, 3, 43)] * 3
    scenes = [grids.scene(s, 50 + i, i % 2 == 1) for i, s in enumerate(shapes)]
    prm = S.default_params(residual=1e-6)
    work = [sc.copy() for sc in scenes]
    _, Ps, P64s = ctx.project_batch(work, prm, pressure64=True)
    for sc, w, bP, bP64 in zip(scenes, work, Ps, P64s):
        one = sc.copy()
        _, P, P64 = ctx.project(one, prm, pressure64=True)
        assert np.array_equal(P, bP) and np.array_equal(P64, bP64)
        assert np.array_equal(w.u, one.u) and np.array_equal(w.v, one.v) and np.array_equal(w.wv, one.wv)


@pytest.mark.parametrize("shape", [(4099, 4, 4), (4098, 8), (30, 40, 20)])
def test_no_liquid(ctx, shape):
    print(f"[gpu-case] no liquid {shape}", flush=True)
    flat = len(shape) == 2
    sc = grids.scene(shape, 3, False)
    sc.fluid[...] = 1.0
    _, P, _ = (ctx.project2d if flat else ctx.project)(sc, S.default_params(residual=1e-6))
    assert not P.any()
    ref = grids.scene(shape, 3, False)
    ref.fluid[...] = 1.0
    A = (O.assemble2 if flat else O.assemble)(ref)
    (O.velocity_update2 if flat else O.velocity_update)(ref, P, A["area"], A["rho"])
    for a, b in zip((sc.u, sc.v) if flat else (sc.u, sc.v, sc.wv), (ref.u, ref.v) if flat else (ref.u, ref.v, ref.wv)):
        assert np.array_equal(a, b)
