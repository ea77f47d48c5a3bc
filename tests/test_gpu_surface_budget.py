"""The surface's device budget against what a run allocates: many particles to a
voxel (the particles' buffers decide), few to many vertices (the grid's), and a
mesh that only its own size puts over the cap."""
import numpy as np
import pytest

from nonnewton_amd import _lib as L
from nonnewton_amd.surface import Surface

pytestmark = pytest.mark.gpu


def need(info, n, anisotropic=True, velocity=False):
    """Bytes of a run: grid, particles, inputs; and those of its mesh."""
    vox, dims = np.prod(info["voxel_dims"]), np.prod(info["dims"])
    grid = 8 * vox + (32 if velocity else 20) * dims + n * (84 + 80 * anisotropic + 12 + 12 * velocity)
    return int(grid), int(info["num_vertices"] * (24 + 12 * velocity) + 12 * info["num_triangles"])


def outcome(x, u, cap, **kw):
    s = Surface(voxel_size=0.04, particle_radius=0.02, velocity=u is not None, **kw)
    s.set_budget(cap)
    try:
        return s.run(x, u)
    except L.NNError as e:
        assert e.code == L.NN_E_OOM
        return None
    finally:
        s.close()


@pytest.mark.parametrize("velocity", [False, True])
def test_dense_particles(velocity):
    rng = np.random.Generator(np.random.PCG64(1))
    cell = np.stack(np.meshgrid(*[np.arange(22)] * 3, indexing="ij"), -1).reshape(-1, 3)
    x = ((np.repeat(cell, 32, 0) + 20 + rng.uniform(0.01, 0.99, (32 * len(cell), 3))) * 0.04).astype(np.float32)
    u = np.ones_like(x) if velocity else None
    info = outcome(x, u, 0, smooth_radius=0.03)
    grid, mesh = need(info, len(x), velocity=velocity)
    counted_before = 8 * np.prod(info["voxel_dims"]) + (72 if velocity else 36) * np.prod(info["dims"]) + 64 * len(x)
    assert counted_before < 0.8 * grid
    assert outcome(x, u, int(0.9 * grid), smooth_radius=0.03) is None
    assert outcome(x, u, grid + mesh + (1 << 20), smooth_radius=0.03) == info


def test_sparse_particles():
    """Two clusters far apart: the vertices between them decide."""
    rng = np.random.Generator(np.random.PCG64(2))
    x = np.concatenate([rng.uniform(0.4, 0.8, (500, 3)), rng.uniform(5.0, 5.4, (500, 3))]).astype(np.float32)
    info = outcome(x, None, 0, smooth_radius=0.1)
    grid, mesh = need(info, len(x))
    assert grid + mesh + (1 << 20) < 30 * np.prod(info["dims"])
    assert outcome(x, None, grid + mesh + (1 << 20), smooth_radius=0.1) == info
    assert outcome(x, None, int(0.95 * grid), smooth_radius=0.1) is None


def test_mesh_over_the_cap():
    rng = np.random.Generator(np.random.PCG64(3))
    x = rng.uniform(0.1, 2.4, (4000, 3)).astype(np.float32)
    info = outcome(x, None, 0, smooth_radius=0.08, isolevel=0.0)
    grid, mesh = need(info, len(x))
    assert mesh > 600000
    assert outcome(x, None, grid + mesh // 2, smooth_radius=0.08) is None
    assert outcome(x, None, grid + mesh + (1 << 20), smooth_radius=0.08) == info
