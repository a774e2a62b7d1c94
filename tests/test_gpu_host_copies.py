"""Host arrays on either side of the size from which several threads copy them: the projection of host arrays
equals the one of the same arrays on the device, bit for bit, outputs included; a batch copies as one.
"""
import numpy as np
import pytest

import shiokaze_amd as S
from shiokaze_amd.devmem import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = S.Context(0)
    yield c
    c.close()


def on_device(ctx, sc, prm):
    arrays = [DeviceArray(a) for a in (sc.fluid, sc.solid, sc.u, sc.v, sc.wv)]
    P = DeviceArray(np.zeros((sc.w, sc.h, sc.d), np.float32))
    f = S.F64 if sc.fluid.dtype == np.float64 else S.F32
    g = S.F64 if sc.solid.dtype == np.float64 else S.F32
    grid = S.Context.device_grid(sc.w, sc.h, sc.d, sc.dt, arrays[0], f, arrays[1], g, arrays[2], arrays[3], arrays[4], pressure=P)
    ctx.project_batch_device([grid], prm)
    out = [a.download() for a in arrays[2:]] + [P.download()]
    for a in arrays + [P]:
        a.free()
    return out


@pytest.mark.parametrize("shape", [(40, 41, 39), (67, 71, 73), (101, 64, 96)])
def test_host_arrays_equal_device_arrays(ctx, shape):
    print(f"[gpu-case] host copies {shape}", flush=True)
    prm = S.default_params(residual=1e-4)
    scenes = [S.make_scene(S.SCENE_DROP_SOLIDS, *shape, seed=s) for s in (1, 2)]
    want = [on_device(ctx, sc, prm) for sc in scenes]
    alone = scenes[0].copy()
    r, P, _ = ctx.project(alone, prm)
    for a, b in zip((alone.u, alone.v, alone.wv, P), want[0]):
        assert np.array_equal(a, b.reshape(a.shape))
    both = [sc.copy() for sc in scenes]
    res, Ps, _ = ctx.project_batch(both, prm)
    for sc, P, w in zip(both, Ps, want):
        for a, b in zip((sc.u, sc.v, sc.wv, P), w):
            assert np.array_equal(a, b.reshape(a.shape))
