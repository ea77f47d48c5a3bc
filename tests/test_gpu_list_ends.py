"""Steps of particles whose lists end around the batches of the 16-lane sweeps
(0, 1, 15, 16, 17, 31, 32, 33, 47, 48 and 49 entries, in clusters far from one
another), with and without surface tension, against the FP32 oracle bit for
bit."""
import numpy as np
import pytest

from nonnewton_amd import scenes
from test_gpu_sweep_lanes import compare

pytestmark = pytest.mark.gpu


def clusters(seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    sc = scenes.tiny_box(seed=seed, fluid_counts=(3, 3, 3), cells=(50, 50, 50), dt=1e-5)
    h = 4.0 * sc.params.particle_radius
    parts = []
    for c, entries in enumerate((0, 1, 15, 16, 17, 31, 32, 33, 47, 48, 49)):
        centre = (np.array([2 + 4 * (c % 4), 2 + 4 * (c // 4), 5]) + 0.5) * h
        parts.append(centre + rng.uniform(-0.28, 0.28, (entries + 1, 3)) * h)
    x = np.concatenate(parts).astype(np.float32)
    sc.x = np.ascontiguousarray(x[rng.permutation(len(x))])
    n = len(x)
    sc.kind = np.zeros(n, np.int32)
    sc.v = rng.uniform(-0.2, 0.2, (n, 3)).astype(np.float32)
    return sc


@pytest.mark.parametrize("seed,surface", [(1, True), (2, False)])
def test_lists_that_end_around_a_batch(seed, surface):
    sc = clusters(seed)
    if not surface:
        sc.params = sc.params.replace(use_surface_tension=False)
    compare(sc, 2)
