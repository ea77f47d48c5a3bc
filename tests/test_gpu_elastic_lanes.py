"""The elastic sweeps with 16 and 4 lanes per member of the stress set against
the FP32 oracle bit for bit: sets below and above a wavefront, and on either
side of the limit between the two forms (32,768)."""
import numpy as np
import pytest

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes
from nonnewton_amd.params import KIND_ELASTIC
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [(1, 1, 1), (3, 7, 3), (5, 13, 1), (32, 32, 32), (32, 32, 33)])
def test_elastic_sweeps(counts):
    sc = scenes.elastic_drop(block_counts=counts, plate_counts=(40, 40))
    rng = np.random.Generator(np.random.PCG64(sum(counts)))
    e = sc.kind == KIND_ELASTIC
    sc.v[e] = rng.uniform(-0.5, 0.5, (int(e.sum()), 3)).astype(np.float32)
    ctx = L.Context(sc.params, sc.n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    o = O.OracleSim.from_scene(sc, precision="f32")
    o.init()
    for _ in range(3):
        ctx.step()
        o.step()
    for fg, fo in [(L.FIELD_X, O.F_X), (L.FIELD_V, O.F_V), (L.FIELD_ACCELERATION, O.F_ACC),
                   (L.FIELD_ROTATION, O.F_ROTATION), (L.FIELD_STRESS, O.F_STRESS)]:
        b = o.get(fo).astype(np.float32)
        a = ctx.download(fg).reshape(b.shape)
        if fo in (O.F_ROTATION, O.F_STRESS):  # held for the elastic particles and their rest neighbors
            a, b = a[e], b[e]
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), fg
    ctx.close()
