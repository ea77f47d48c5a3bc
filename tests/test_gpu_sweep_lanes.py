"""The list sweeps with 1, 4 and 16 lanes per particle and their shortened
divisions and square roots, against the FP32 oracle bit for bit: scene sizes on
both sides of the lane limits, unjittered lattices (zero components),
coincident and nearly coincident particles, components around the smallest
normal floats and negative zeros, and a kernel radius outside the range the
shortened forms hold for."""
import numpy as np
import pytest

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu

FIELDS = [("x", L.FIELD_X, O.F_X), ("v", L.FIELD_V, O.F_V), ("acceleration", L.FIELD_ACCELERATION, O.F_ACC),
          ("volume", L.FIELD_VOLUME, O.F_VOLUME), ("density", L.FIELD_DENSITY, O.F_DENSITY),
          ("dfsph_factor", L.FIELD_DFSPH_FACTOR, O.F_DFSPH_FACTOR), ("density_adv", L.FIELD_DENSITY_ADV, O.F_DENSITY_ADV)]


def compare(sc, steps):
    ctx = L.Context(sc.params, sc.n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    o = O.OracleSim.from_scene(sc, precision="f32")
    o.init()
    for k in range(steps):
        sg, so = ctx.step(), o.step()
        assert sg["num_pairs"] == so["num_pairs"]
        assert sg["max_density"] == so["max_density"]
        assert (sg["iterations_v"], sg["iterations_p"]) == (so["iterations_v"], so["iterations_p"])
    for name, fg, fo in FIELDS:
        b = o.get(fo)
        a = ctx.download(fg).reshape(b.shape).astype(b.dtype)
        # bits, so that a zero's sign counts
        assert np.array_equal(a.astype(np.float32).view(np.uint32), b.astype(np.float32).view(np.uint32)), name
    nbr, cnt = ctx.neighbors()
    on, oc = o.neighbors()
    assert np.array_equal(cnt, oc)
    assert np.array_equal(nbr[:, : on.shape[1]], on)
    ctx.close()


# slots in use: about 1,000, 2,600, 32,768 on either side, and above 196,608
@pytest.mark.parametrize("counts,cells,compensated", [
    ((3, 5, 3), (12, 14, 12), True), ((8, 9, 7), (18, 20, 18), False), ((29, 26, 25), (50, 50, 38), True),
    ((31, 27, 25), (50, 50, 38), False), ((60, 50, 50), (92, 72, 88), True)])
def test_sizes_on_both_sides_of_the_lane_limits(counts, cells, compensated):
    sc = scenes.tiny_box(seed=3, fluid_counts=counts, cells=cells, compensated=compensated, dt=5e-4)
    rng = np.random.Generator(np.random.PCG64(4))
    f = sc.kind == 0
    sc.v[f] = rng.uniform(-0.5, 0.5, (int(f.sum()), 3)).astype(np.float32)
    compare(sc, 2)


def test_zero_tiny_and_coincident_components():
    sc = scenes.tiny_box(seed=5, fluid_counts=(6, 6, 6), cells=(14, 14, 14), boundary_viscosity=0.02)
    f = np.flatnonzero(sc.kind == 0)
    sc.x[f] = scenes.lattice((0.06, 0.06, 0.06), (6, 6, 6)).astype(np.float32)  # exact lattice: zero components
    sc.x[f[1]] = sc.x[f[0]]                                                     # coincident
    sc.x[f[3]] = sc.x[f[2]] + np.float32(3e-6)                                  # closer than 1e-5
    # a column of particles on the domain's face: x differs by zeros of both
    # signs and by denormal and tiny amounts
    for k, t in enumerate([0.0, -0.0, 1e-45, 3e-39, 1e-36, 2e-31, 7e-31, 1e-30]):
        sc.x[f[40 + k]] = (np.float32(t), np.float32(0.06 + 0.013 * k), np.float32(0.06))
    sc.v[f, 0] = -0.0
    sc.v[f[::2], 1] = 0.1
    compare(sc, 1)


@pytest.mark.parametrize("scale", [2.0 ** -16, 2.0 ** -15, 2.0 ** 24])
def test_kernel_radius_outside_the_midrange(scale):
    """h = 0.04 scale: below 2^-20 (plain forms), just above it, and 2^19."""
    sc = scenes.tiny_box(seed=6, fluid_counts=(5, 6, 5), cells=(12, 14, 12))
    p = sc.params
    sc.params = p.replace(domain_end=tuple(float(np.float32(c * scale)) for c in p.domain_end),
                          particle_radius=p.particle_radius * scale, gravity=(0.0, -9.81 * scale, 0.0))
    sc.x = (sc.x * np.float32(scale)).astype(np.float32)
    rng = np.random.Generator(np.random.PCG64(7))
    f = sc.kind == 0
    sc.v[f] = (rng.uniform(-0.5, 0.5, (int(f.sum()), 3)) * scale).astype(np.float32)
    compare(sc, 1)
