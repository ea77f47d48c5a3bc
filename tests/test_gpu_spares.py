"""A pool's memory used again by later scenes: rounds of admissions, ticks and
retirements of scenes of several sizes and kinds (cold and warm solves, an
elastic block, more particles than are uploaded through pinned memory), with
room for spare blocks and with so small a budget that most are freed; every
scene ends with the bits it has alone in a context."""
import numpy as np
import pytest

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes

pytestmark = pytest.mark.gpu

FIELDS = (L.FIELD_X, L.FIELD_V, L.FIELD_VISC_DIFF)


def make(k):
    if k == 2:
        return scenes.elastic_drop(block_counts=(5, 4, 6), plate_counts=(16, 16))
    if k == 3:
        return scenes.tiny_box(seed=3, fluid_counts=(24, 40, 42), cells=(34, 50, 52), dt=5e-4)  # 40,320 + walls
    sc = scenes.tiny_box(seed=k, fluid_counts=(5 + k, 6, 5), cells=(16 + k, 14, 12), use_non_newtonian=True,
                         non_newton_method=1, consistency_index=20.0, power_index=0.7, max_viscosity=1e4,
                         viscosity_method=1, weiler_tol=1e-4, dt=5e-4, warm_start=k % 2)
    f = sc.kind == 0
    sc.v[f] = np.random.Generator(np.random.PCG64(k)).uniform(-0.2, 0.2, (int(f.sum()), 3)).astype(np.float32)
    return sc


def alone(sc, steps):
    ctx = L.Context(sc.params, sc.n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    for _ in range(steps):
        ctx.step()
    out = [ctx.download(f).copy() for f in FIELDS]
    ctx.close()
    return out


@pytest.mark.parametrize("budget", [1 << 30, 200 << 20])
def test_memory_is_used_again(budget):
    scs = [make(k) for k in range(5)]
    want = [alone(sc, 3) for sc in scs]
    pool = L.Pool(budget)
    rng = np.random.Generator(np.random.PCG64(7))
    for _ in range(5):
        order = rng.permutation(5)
        slots = {int(k): pool.admit(scs[k].params, scs[k].x, scs[k].kind, scs[k].v) for k in order}
        assert all(s is not None for s in slots.values())
        for _ in range(3):
            pool.tick()
        for k, s in slots.items():
            for f, w in zip(FIELDS, want[k]):
                assert np.array_equal(pool.read(s, f).reshape(-1), w.reshape(-1)), (k, f)
            pool.retire(s)
    pool.close()
