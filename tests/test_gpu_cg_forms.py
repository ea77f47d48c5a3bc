"""Which form a Weiler solve takes, and the way back from the one-launch form: a
solve that leaves after 0, 1, 2 or 5 exchanges is repeated with the two-launch
form and gives that form's bits, iteration counts and status."""
import threading

import numpy as np
import pytest

from nonnewton_amd import _lib as L
from test_gpu_cg_solve import column

pytestmark = pytest.mark.gpu


def run(sc, steps=3, depth=0, patience=-1):
    ctx = L.Context(sc.params, sc.n)
    ctx.set_kernel_depth("cg_matvec", depth)
    ctx.set_cg_patience(patience)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    its = []
    for _ in range(steps):
        st = ctx.step()
        its.append((st["iterations_cg"], st["iterations_p"], st["cg_rel_residual"], st["status"]))
    out = [ctx.download(f) for f in (L.FIELD_X, L.FIELD_V, L.FIELD_VISC_DIFF, L.FIELD_ACCELERATION)]
    forms = ctx.cg_forms()
    ctx.close()
    return its, out, forms


def cut(sc, waves):
    keep = waves * 64 - 3
    fluid, wall = np.flatnonzero(sc.kind == 0), np.flatnonzero(sc.kind != 0)
    idx = np.concatenate([fluid, wall])[:keep]
    sc.x, sc.v, sc.kind = sc.x[idx], sc.v[idx], sc.kind[idx]
    assert -(-len(idx) // 64) == waves
    return sc


@pytest.mark.parametrize("waves", [1, 40, 256, 257])
def test_form_by_size(waves):
    sc = cut(column((22, 30, 20), (40, 40, 40)) if waves > 1 else column((3, 6, 3), (12, 12, 12)), waves)
    assert run(sc)[2] == ((3, 0, 0) if waves <= 256 else (0, 3, 0))
    assert run(sc, depth=2)[2] == (0, 3, 0)


@pytest.mark.parametrize("warm", [0, 1])
@pytest.mark.parametrize("counts,cells", [((6, 6, 6), (14, 14, 14)), ((13, 19, 11), (30, 30, 20))])
@pytest.mark.parametrize("patience", [0, 1, 2, 5])
def test_way_back(patience, counts, cells, warm):
    sc = column(counts, cells, warm_start=warm)
    ia, a, fa = run(sc, depth=2)
    ib, b, fb = run(sc, patience=patience)
    assert max(i for i, _, _, _ in ia) > 6
    assert fa == (0, 3, 0) and fb[0] == 0 and fb[1] == 3 and fb[2] >= 1
    assert ia == ib
    assert all(np.array_equal(p, q) for p, q in zip(a, b))


@pytest.mark.parametrize("patience", [0, 3])
def test_way_back_at_the_iteration_limit(patience):
    sc = column((10, 10, 10), (20, 20, 20), weiler_max_iter=5, weiler_tol=1e-7)
    ia, a, _ = run(sc, depth=2)
    ib, b, forms = run(sc, patience=patience)
    assert all(i == 5 and s & 32 for i, _, _, s in ia) and forms[2] >= 1
    assert ia == ib and all(np.array_equal(p, q) for p, q in zip(a, b))


def test_tried_again_later():
    """A solve left once is tried again after 256 others."""
    sc = column((4, 4, 4), (10, 10, 10))
    ctx = L.Context(sc.params, sc.n)
    ctx.set_cg_patience(0)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    ctx.step()
    assert ctx.cg_forms() == (0, 1, 1)
    ctx.set_cg_patience(-1)
    ctx.step(256)
    assert ctx.cg_forms() == (0, 257, 1)
    ctx.step(3)
    assert ctx.cg_forms() == (3, 257, 1)
    ctx.close()


@pytest.mark.parametrize("waves", [(200, 200, 200), (200, 40, 120)])
def test_contexts_in_threads(waves):
    """Contexts stepped at once from their own threads, with more waves in all
    than the device has compute units: the bits of each alone, and no solve
    begun in one launch that had to be left."""
    scs = [cut(column((22, 30, 20), (40, 40, 40)), w) for w in waves]
    want = [run(sc, 40) for sc in scs]
    got = [None] * len(scs)
    start = threading.Barrier(len(scs))

    def work(k):
        start.wait()
        got[k] = run(scs[k], 40)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(scs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for (ia, a, _), (ib, b, forms) in zip(want, got):
        assert ia == ib and all(np.array_equal(p, q) for p, q in zip(a, b))
        assert forms[0] + forms[1] == 40 and forms[2] == 0
