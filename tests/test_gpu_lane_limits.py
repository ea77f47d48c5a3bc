"""Either side of the slots at which a sweep's number of lanes changes (16,384
for density and strain, 98,304 for density, 196,608 for the non-pressure sweep
without velocity terms, 16,384 members for the rotations): bits of the FP32
oracle, and a boundary viscosity that is set while one lane runs."""
import numpy as np
import pytest

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes
from oracle import oracle as O
from test_gpu_elastic_lanes import test_elastic_sweeps as elastic_sweeps
from test_gpu_sweep_lanes import compare

pytestmark = pytest.mark.gpu


def cut(sc, n):
    """The scene with its first n particles (fluid first)."""
    sc.x, sc.v, sc.kind = sc.x[:n], sc.v[:n], sc.kind[:n]
    assert len(sc.x) == n
    rng = np.random.Generator(np.random.PCG64(n))
    f = sc.kind == 0
    sc.v[f] = rng.uniform(-0.3, 0.3, (int(f.sum()), 3)).astype(np.float32)
    return sc


@pytest.mark.parametrize("slots,counts,cells", [(16384, (24, 24, 20), (40, 40, 38)), (98304, (48, 40, 44), (76, 62, 64))])
@pytest.mark.parametrize("more", [0, 1])
def test_explicit(slots, counts, cells, more):
    compare(cut(scenes.tiny_box(seed=3, fluid_counts=counts, cells=cells, dt=5e-4, use_non_newtonian=True,
                                non_newton_method=0, viscosity0=0.02), slots + more), 2)


def box(n, **kw):
    return cut(scenes.tiny_box(seed=4, fluid_counts=(60, 52, 52), cells=(92, 76, 90), dt=5e-4, viscosity_method=1,
                               weiler_max_iter=2, viscosity=0.02, **kw), n)


@pytest.mark.parametrize("n", [196608, 196609])
def test_implicit(n):
    """Two CG iterations, so that the sums of the implicit solve stay those of
    the oracle's order only to rounding: densities and lists, which the sweeps
    before it give, in bits, positions and velocities to the solve's."""
    sc = box(n)
    ctx = L.Context(sc.params, sc.n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    o = O.OracleSim.from_scene(sc, precision="f32")
    o.init()
    assert ctx.step()["num_pairs"] == o.step()["num_pairs"]
    b = o.get(O.F_DENSITY)
    assert np.array_equal(ctx.download(L.FIELD_DENSITY).astype(b.dtype), b)
    for fg, fo in ((L.FIELD_X, O.F_X), (L.FIELD_V, O.F_V)):
        b = o.get(fo)
        assert np.abs(ctx.download(fg).reshape(b.shape) - b).max() <= 1e-5 * np.abs(b).max()
    ctx.close()


def test_boundary_viscosity_set_between_steps():
    out = []
    for made_with in (0.0, 0.05):
        sc = box(196700, boundary_viscosity=made_with)
        ctx = L.Context(sc.params, sc.n)
        ctx.upload(sc.x, sc.kind, sc.v)
        ctx.init()
        ctx.set_param("boundary_viscosity", 0.05)
        ctx.step(2)
        out.append([ctx.download(f) for f in (L.FIELD_X, L.FIELD_V)])
        ctx.close()
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    sc = box(196700)
    ctx = L.Context(sc.params, sc.n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    ctx.step(2)
    assert not np.array_equal(ctx.download(L.FIELD_V), out[0][1])
    ctx.close()


@pytest.mark.parametrize("counts", [(32, 32, 16), (32, 32, 17)])
def test_rotations(counts):
    elastic_sweeps(counts)
