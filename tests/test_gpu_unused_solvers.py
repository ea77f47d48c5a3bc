"""Statistics of a scene that uses neither the divergence nor the implicit solver:
zeros, also in a pool where a scene that used both has just left its place."""
import pytest

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes

pytestmark = pytest.mark.gpu


def test_counts_of_unused_solvers():
    both = scenes.tiny_box(seed=1, fluid_counts=(6, 8, 6), cells=(16, 16, 14), use_non_newtonian=True, non_newton_method=1,
                           consistency_index=20.0, power_index=0.7, max_viscosity=1e4, viscosity_method=1,
                           weiler_tol=1e-4, dt=5e-4)
    both.v[both.kind == 0, 0] = 0.3
    none = scenes.tiny_box(seed=2, enable_divergence_solver=False)
    pool = L.Pool(1 << 30)
    a = pool.admit(both.params, both.x, both.kind, both.v)
    b = pool.admit(none.params, none.x, none.kind, none.v)
    for _ in range(2):
        pool.tick()
    assert pool.stats(a)["iterations_v"] > 0 and pool.stats(a)["iterations_cg"] > 0
    for leave in (False, True):
        if leave:
            pool.retire(a)
            pool.tick()
        st = pool.stats(b)
        assert (st["iterations_v"], st["iterations_cg"], st["avg_density_err_v"], st["cg_rel_residual"]) == (0, 0, 0.0, 0.0)
        assert st["iterations_p"] > 0
    pool.close()
