"""The face kernels of a time step (extrapolation, constraint, advection) at the edges of their work units: rows
around a word of 32 faces, wavefronts of 64, index division at extents of 2 to 146, and a field large
enough that a wavefront takes eight groups of faces, with a ragged end.  Random activity, dense and sparse; every
value equal to the oracle's, bit for bit.
"""
import numpy as np
import pytest

import shiokaze_amd as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (5, 4, 31), (3, 7, 32), (4, 3, 33), (9, 2, 64), (2, 65, 3), (139, 143, 146)]


@pytest.fixture(scope="module")
def ctx():
    c = S.Context(0)
    yield c
    c.close()


def field(shape, density, seed):
    rng = np.random.default_rng(seed)
    shapes = O.face_shapes(*shape)
    vel = [rng.normal(size=s).astype(np.float32) for s in shapes]
    act = [(rng.uniform(size=s) < density).astype(np.uint8) for s in shapes]
    solid = (rng.normal(size=tuple(n + 1 for n in shape)) + 0.5).astype(np.float32)
    fluid = rng.normal(size=shape).astype(np.float32) * 0.1
    return vel, act, solid, fluid


def assert_same(got, want):
    for a, (x, y) in enumerate(zip(got, want)):
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), a


@pytest.mark.parametrize("density", [0.03, 0.6])
@pytest.mark.parametrize("shape", SHAPES)
def test_face_kernels_match_oracle(ctx, shape, density):
    print(f"[gpu-case] faces {shape} density={density}", flush=True)
    vel, act, solid, fluid = field(shape, density, sum(shape))
    vg, ag = [v.copy() for v in vel], [a.copy() for a in act]
    ctx.extrapolate_velocity(*shape, vg, ag, solid=solid, width=2, constrain=True)
    vo, ao = [v.copy() for v in vel], [a.copy() for a in act]
    O.extrapolate(*shape, vo, ao, 2)
    O.constrain_velocity(*shape, vo, ao, solid)
    assert_same(vg, vo)
    assert_same(ag, ao)
    dt = 0.4 / max(shape)  # a few cells for the fastest of the random values
    for mc in (True, False):
        vg, vo = [v.copy() for v in vel], [v.copy() for v in vel]
        ctx.advect_velocity(*shape, vg, act, fluid, dt, maccormack=mc)
        O.advect_velocity(*shape, vo, act, fluid, dt, maccormack=mc)
        assert_same(vg, vo)
