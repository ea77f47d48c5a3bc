"""A surface's arrays on either side of the size that crosses through pinned
memory (1 MiB together): particles and velocities going in, a mesh with and
without normals and its velocities coming out, and runs of different sizes one
after the other, against the oracle bit for bit."""
import numpy as np
import pytest

from nonnewton_amd.surface import Surface
from oracle import surface as O

pytestmark = pytest.mark.gpu


def block(n, seed):
    a = max(1, int(round(n ** (1 / 3))))
    k = np.arange(n)
    x = np.stack([k // (a * a), k // a % a, k % a], 1) * 0.02 + 0.21
    return (x + np.random.Generator(np.random.PCG64(seed)).uniform(-0.003, 0.003, x.shape)).astype(np.float32)


@pytest.mark.parametrize("normals", [True, False])
def test_transfers(normals):
    # 24 n bytes in: 43,690 particles are 1 MiB
    kw = dict(voxel_size=0.02, particle_radius=0.02, smooth_radius=0.04, normals=normals)
    s = Surface(velocity=True, **kw)
    for n in (1, 43690, 43691, 700):
        x = block(n, n)
        u = np.random.Generator(np.random.PCG64(n + 1)).uniform(-1, 1, x.shape).astype(np.float32)
        s.run(x, u)
        o = O.reconstruct(x, velocity=u, **kw)
        v, f, m = s.mesh()
        assert np.array_equal(v, o["vertices"]) and np.array_equal(f, o["faces"])
        if normals:
            assert np.array_equal(m, o["normals"])
        assert np.array_equal(s.mesh_velocity(), o["mesh_velocity"])
    s.close()


@pytest.mark.parametrize("voxel", [0.012, 0.006])
def test_mesh_sizes(voxel):
    """Meshes of below and above 1 MiB."""
    kw = dict(voxel_size=voxel, particle_radius=0.02, smooth_radius=0.04, normals=True)
    x = block(9000, 3)
    s = Surface(**kw)
    s.run(x)
    o = O.reconstruct(x, **kw)
    v, f, m = s.mesh()
    size = v.nbytes + f.nbytes + m.nbytes
    assert (size > 1 << 20) == (voxel == 0.006)
    assert np.array_equal(v, o["vertices"]) and np.array_equal(f, o["faces"]) and np.array_equal(m, o["normals"])
    s.close()
