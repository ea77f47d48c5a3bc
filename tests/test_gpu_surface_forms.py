"""The smooth field's FP64 tile sums and the contour over compacted cubes against
the oracle bit for bit: velocities whose sums fit and whose sums take the
general form, a smooth radius below the range of the short poly6 quotient, cube
counts around a workgroup's 64, and a voxel grid whose scan needs its block sums
scanned first (more than 2^25 voxels)."""
import numpy as np
import pytest

from nonnewton_amd.surface import Surface
from oracle import surface as O

pytestmark = pytest.mark.gpu


def check(x, vel=None, **kw):
    s = Surface(velocity=vel is not None, **kw)
    info = s.run(x, vel)
    o = O.reconstruct(x, velocity=vel, **kw)
    assert np.array_equal(s.field(1), o["field"], equal_nan=True)
    v, f, n = s.mesh()
    assert np.array_equal(v, o["vertices"]) and np.array_equal(f, o["faces"])
    if kw.get("normals"):
        assert np.array_equal(n, o["normals"])
    if vel is not None:
        assert np.array_equal(s.mesh_velocity(), o["mesh_velocity"])
    s.close()
    return o


def block(n, seed, sp):
    a = max(1, int(round(n ** (1 / 3))))
    k = np.arange(n)
    x = np.stack([k // (a * a), k // a % a, k % a], 1) * sp + 10.5 * sp
    return (x + np.random.Generator(np.random.PCG64(seed)).uniform(-0.15 * sp, 0.15 * sp, x.shape)).astype(np.float32)


@pytest.mark.parametrize("scale,sp", [(1.0, 0.02), (1e7, 0.02), (1.0, 0.0016)])
def test_velocity_sums(scale, sp):
    """h = 0.05 and 0.004 (h^9 below 2^-63)."""
    x = block(600, 3, sp)
    u = (scale * np.random.Generator(np.random.PCG64(4)).uniform(-1, 1, x.shape)).astype(np.float32)
    small = sp < 0.01  # no negative values there: nothing to smooth by
    o = check(x, u, voxel_size=sp / 2, particle_radius=sp, smooth_radius=2.5 * sp, normals=True,
              isolevel=0.2 if small else 0.0, smooth_iterations=0 if small else 1)
    assert np.any(o["mesh_velocity"] != 0)


@pytest.mark.parametrize("voxel", [0.05, 0.045, 0.04, 0.036, 0.03])
def test_few_cubes(voxel):
    o = check(block(27, 7, 0.04), voxel_size=voxel, particle_radius=0.04, smooth_radius=0.1, normals=True)
    assert len(o["vertices"]) > 0


def test_more_voxels_than_one_scan_level():
    x = np.concatenate([block(50, 9, 0.02), block(50, 10, 0.02) + np.float32(3.3)])
    check(x, voxel_size=0.01, particle_radius=0.02, smooth_radius=0.04)
