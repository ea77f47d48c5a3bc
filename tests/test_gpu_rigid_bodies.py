"""Rigid bodies projected by one workgroup each, and beyond that size by one
launch per stage, against the FP32 oracle bit for bit: one particle, a wavefront
and one more, the largest body of the one-launch form (4,096 particles) and one
above, with a second body that starts below the padding height."""
import numpy as np
import pytest

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes
from nonnewton_amd.params import SceneParams
from oracle import oracle as O

pytestmark = pytest.mark.gpu
SP = scenes.SPACING


@pytest.mark.parametrize("counts,coupling", [((1, 1, 1), 1), ((4, 4, 4), 2), ((5, 13, 1), 2), ((16, 16, 16), 2),
                                             ((16, 16, 17), 2)])
def test_bodies_around_the_one_launch_limit(counts, coupling):
    rng = np.random.Generator(np.random.PCG64(31))
    cells = (40, 40, 40)
    p = SceneParams(domain_end=tuple(c * SP for c in cells), gravity=(0.0, -9.81, 0.0), dt=5e-4,
                    coupling_interval=coupling)
    fluid = scenes.jitter(rng, scenes.lattice((6 * SP, 3 * SP, 6 * SP), (8, 6, 8)))
    low = scenes.lattice((30 * SP, 1.2 * SP, 30 * SP), (4, 4, 4))
    body = scenes.lattice((9 * SP, 12 * SP, 9 * SP), counts)
    sc = scenes.assemble("bodies", p, fluid, scenes.shell(cells), None, 1, rigid=[low, body])
    ctx = L.Context(sc.params, sc.n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    o = O.OracleSim.from_scene(sc, precision="f32")
    o.init()
    for _ in range(6):
        ctx.step()
        o.step()
    for fg, fo in [(L.FIELD_X, O.F_X), (L.FIELD_V, O.F_V), (L.FIELD_ACCELERATION, O.F_ACC)]:
        b = o.get(fo).astype(np.float32)
        assert np.array_equal(ctx.download(fg).reshape(b.shape).view(np.uint32), b.view(np.uint32)), fg
    ctx.close()
