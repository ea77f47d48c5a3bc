"""A small scene's CG in one launch against the CG as two launches an iteration
(which a gather depth asked for selects), bit for bit with the same iteration
counts: one wave to the most waves of one launch and one more, lists of up to
48 entries and more, with and without the warm start, and a solve that ends at
its iteration limit."""
import numpy as np
import pytest

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes

pytestmark = pytest.mark.gpu


def runs(sc, steps):
    out = []
    for depth in (0, 2):
        ctx = L.Context(sc.params, sc.n)
        ctx.set_kernel_depth("cg_matvec", depth)
        ctx.upload(sc.x, sc.kind, sc.v)
        ctx.init()
        its = []
        for _ in range(steps):
            st = ctx.step()
            its.append((st["iterations_cg"], st["cg_rel_residual"], st["status"]))
        out.append((its, ctx.download(L.FIELD_X), ctx.download(L.FIELD_V), ctx.download(L.FIELD_VISC_DIFF)))
        ctx.close()
    (ia, *a), (ib, *b) = out
    assert ia == ib
    assert all(np.array_equal(p, q) for p, q in zip(a, b))
    return ia


def column(counts, cells, **kw):
    p = dict(use_non_newtonian=True, non_newton_method=1, consistency_index=20.0, power_index=0.7, max_viscosity=1e4,
             viscosity_method=1, weiler_tol=1e-4, dt=5e-4)
    p.update(kw)
    sc = scenes.tiny_box(seed=9, fluid_counts=counts, cells=cells, **p)
    f = sc.kind == 0
    sc.v[f] = np.random.Generator(np.random.PCG64(10)).uniform(-0.3, 0.3, (int(f.sum()), 3)).astype(np.float32)
    return sc


@pytest.mark.parametrize("counts,cells", [((6, 6, 6), (14, 14, 14)), ((13, 19, 11), (30, 30, 20)), ((20, 20, 20), (34, 34, 34))])
@pytest.mark.parametrize("warm", [0, 1])
def test_sizes(counts, cells, warm):
    assert max(i for i, _, _ in runs(column(counts, cells, warm_start=warm), 4)) > 3


@pytest.mark.parametrize("waves", [1, 255, 256, 257])
def test_wave_limits(waves):
    """Scenes cut to exactly `waves` waves of slots (the last one partly used)."""
    sc = column((22, 30, 20), (40, 40, 40)) if waves > 1 else column((3, 6, 3), (12, 12, 12))
    keep = waves * 64 - 3
    fluid = np.flatnonzero(sc.kind == 0)
    wall = np.flatnonzero(sc.kind != 0)
    idx = np.concatenate([fluid[: min(len(fluid), keep)], wall])[:keep]
    sc.x, sc.v, sc.kind = sc.x[idx], sc.v[idx], sc.kind[idx]
    assert -(-len(idx) // 64) == waves
    runs(sc, 3)


def test_long_lists():
    sc = column((8, 10, 8), (18, 22, 18), particle_radius=0.0118)
    ctx = L.Context(sc.params, sc.n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    assert ctx.download(L.FIELD_NUM_NEIGHBORS)[sc.kind == 0].max() > 48
    ctx.close()
    runs(sc, 3)


def test_iteration_limit():
    its = runs(column((10, 10, 10), (20, 20, 20), weiler_max_iter=5, weiler_tol=1e-7), 3)
    assert all(i == 5 for i, _, _ in its)
