"""The anisotropy's neighbor lists against the oracle bit for bit where they
branch: more neighbors than a list holds (1,024), a list that is exactly full,
columns with more candidates than are laid out at a time, and neighbors farther
apart in the sorted order than a list entry reaches (65,535)."""
import numpy as np
import pytest

from nonnewton_amd.surface import Surface
from oracle import surface as O

pytestmark = pytest.mark.gpu


def check(x, **kw):
    s = Surface(**kw)
    s.run(x)
    o = O.reconstruct(x, **kw)
    G, xb = s.aniso()
    assert np.array_equal(G, o["G"], equal_nan=True) and np.array_equal(xb, o["xbar"])
    assert np.array_equal(s.field(0), o["field0"])
    s.close()


@pytest.mark.parametrize("n", [960, 961, 1024, 1025, 2500])
def test_full_lists(n):
    """A cloud of which every particle is every other's neighbor."""
    rng = np.random.Generator(np.random.PCG64(n))
    x = (0.5 + rng.uniform(-0.025, 0.025, (n, 3))).astype(np.float32)
    check(x, voxel_size=0.01, particle_radius=0.02, smooth_radius=0.06)


def test_long_columns():
    """Up to 60 particles a voxel along z."""
    rng = np.random.Generator(np.random.PCG64(5))
    x = np.stack([0.505 + rng.uniform(-0.004, 0.004, 700), 0.505 + rng.uniform(-0.004, 0.004, 700),
                  0.4 + 0.13 * (np.arange(700) / 700)], 1).astype(np.float32)
    check(x, voxel_size=0.01, particle_radius=0.02, smooth_radius=0.06)


def test_neighbors_far_apart_in_the_sorted_order():
    """Sheets of 68,121 particles, one after the other in the order."""
    k = np.arange(261)
    sheet = np.stack(np.meshgrid([0.0], k, k, indexing="ij"), -1).reshape(-1, 3)
    x = np.concatenate([sheet, sheet + [1, 0, 0]]) * 0.02 + 0.3
    x = x + np.random.Generator(np.random.PCG64(6)).uniform(-0.003, 0.003, x.shape)
    check(x.astype(np.float32), voxel_size=0.02, particle_radius=0.02, smooth_radius=0.03)
