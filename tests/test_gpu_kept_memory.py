"""The memory that pools keep for their next scenes: bounded over all lanes of a
budget, within the budget together with the scenes, given back when an
allocation of another object fails and when the last pool goes."""
import numpy as np
import pytest
import torch

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes
from nonnewton_amd.lanes import LanePool
from nonnewton_amd.params import SceneParams

pytestmark = pytest.mark.gpu


def block(counts):
    """A lattice of fluid in a box with some room."""
    x = scenes.lattice((0.06, 0.06, 0.06), counts).astype(np.float32)
    p = SceneParams(domain_end=tuple(0.02 * (c + 6) for c in counts), dt=5e-4)
    return p, x, np.zeros(len(x), np.int32)


def test_one_bound_for_all_lanes():
    scene = block((48, 64, 64))  # 150 MB
    lp = LanePool(2 << 30, lanes=3)
    fp = lp.footprint(scene[0], len(scene[1]))
    bound = (2 << 30) // 8
    assert bound / 2 < fp < bound
    for _ in range(3):
        keys = [lp.admit(*scene) for _ in range(3)]
        assert {k[0] for k in keys} == {0, 1, 2}
        assert L.pool_kept_bytes() <= bound
        lp.tick_all()
        for k in keys:
            lp.retire(k)
        lp.tick_all()
    other = L.Pool(1 << 30)
    assert other.admit(*block((8, 8, 8))) is not None
    assert 0 < L.pool_kept_bytes() <= bound
    lp.close()
    assert L.pool_kept_bytes() <= (1 << 30) // 8
    other.close()
    assert L.pool_kept_bytes() == 0


def test_scenes_and_kept_memory_within_the_budget():
    """A pool filled to its budget keeps nothing beside its scenes."""
    scene = block((24, 32, 32))
    probe = L.Pool(1 << 30)
    fp = probe.footprint(scene[0], len(scene[1]))
    probe.close()
    budget = 9 * fp
    pool = L.Pool(budget)
    slots = []
    for _ in range(8):
        slots.append(pool.admit(*scene))
        pool.tick()
        in_use = pool.info()[2]
        assert L.pool_kept_bytes() <= max(0, min(budget // 8, budget - in_use))
    assert None not in slots and pool.admit(*scene) is None
    pool.close()


def test_another_objects_allocation_takes_it():
    """With the device's memory full but for 0.4 GB, a context that needs 0.6
    gets the 0.7 GB that a pool keeps."""
    pool = L.Pool(8 << 30)
    big = block((96, 96, 96))
    slot = pool.admit(*big)
    pool.tick()
    pool.retire(slot)
    small = block((8, 8, 8))
    assert pool.admit(*small) is not None
    assert L.pool_kept_bytes() > 600 << 20
    need = block((80, 96, 96))
    ctx = L.Context(need[0], len(need[1]))
    rest = []
    for left in (2 << 30, 400 << 20):  # the free bytes are told exactly only once most are taken
        rest.append(torch.empty(torch.cuda.mem_get_info()[0] - left, dtype=torch.uint8, device="cuda"))
    try:
        ctx.upload(need[1], need[2])
        assert L.pool_kept_bytes() == 0
    finally:
        del rest
        torch.cuda.empty_cache()
        ctx.close()
        pool.close()
