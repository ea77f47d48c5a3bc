"""Fields cross between cell order on the device and original order in host
memory: uploads and downloads of each three-component field of scenes whose
original order is unlike cell order, 227, 256 (one workgroup) and 259 particles,
bit for bit (NaN payloads included)."""
import numpy as np
import pytest

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def scene(counts, seed):
    sc = scenes.tiny_box(seed=seed, fluid_counts=counts, cells=(14, 6, 6), dt=5e-4)
    rng = np.random.Generator(np.random.PCG64(seed))
    order = rng.permutation(sc.n)  # original order unlike cell order
    sc.x, sc.kind = np.ascontiguousarray(sc.x[order]), np.ascontiguousarray(sc.kind[order])
    sc.v = rng.uniform(-0.1, 0.1, (sc.n, 3)).astype(np.float32) * (sc.kind == 0)[:, None].astype(np.float32)
    return sc


@pytest.mark.parametrize("counts,n", [((1, 1, 1), 227), ((5, 3, 2), 256), ((11, 3, 1), 259)])
def test_fields_keep_their_order(counts, n):
    sc = scene(counts, 11)
    assert sc.n == n
    ctx = L.Context(sc.params, sc.n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    o = O.OracleSim.from_scene(sc, precision="f32")
    o.init()
    ctx.step()
    o.step()
    for fg, fo in [(L.FIELD_X, O.F_X), (L.FIELD_V, O.F_V), (L.FIELD_ACCELERATION, O.F_ACC)]:
        b = o.get(fo).astype(np.float32)
        assert np.array_equal(ctx.download(fg).reshape(b.shape).view(np.uint32), b.view(np.uint32))
    marks = (np.arange(3 * sc.n, dtype=np.uint32) * 2654435761 & 0x7FFFFFFF).reshape(-1, 3)  # any bits
    for f in (L.FIELD_V, L.FIELD_VISC_DIFF):
        before = ctx.download(L.FIELD_X)
        ctx.upload_field(f, marks.view(np.float32))
        assert np.array_equal(ctx.download(f).reshape(-1, 3).view(np.uint32), marks)
        assert np.array_equal(ctx.download(L.FIELD_X), before)
    # the volumes beside the positions are kept
    volume = ctx.download(L.FIELD_VOLUME)
    ctx.upload_field(L.FIELD_X, marks.view(np.float32))
    assert np.array_equal(ctx.download(L.FIELD_X).reshape(-1, 3).view(np.uint32), marks)
    assert np.array_equal(ctx.download(L.FIELD_VOLUME), volume)
    ctx.close()


@pytest.mark.parametrize("n", [87380, 87381, 87382])
def test_fields_on_either_side_of_the_staging_size(n):
    """1 MiB of a field is 87,381 particles."""
    sc = scenes.tiny_box(seed=2, fluid_counts=(3, 3, 3), cells=(100, 100, 100))
    rng = np.random.Generator(np.random.PCG64(n))
    x = scenes.lattice((0.1, 0.1, 0.1), (45, 45, 45)).astype(np.float32)
    sc.x = np.ascontiguousarray(x[rng.permutation(len(x))[:n]])
    sc.kind, sc.v = np.zeros(n, np.int32), np.zeros((n, 3), np.float32)
    ctx = L.Context(sc.params, sc.n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()  # the slots are in cell order now
    assert np.array_equal(ctx.download(L.FIELD_X).reshape(-1, 3), sc.x)
    marks = (np.arange(3 * n, dtype=np.uint32) * 2654435761 & 0x7FFFFFFF).reshape(-1, 3)
    ctx.upload_field(L.FIELD_V, marks.view(np.float32))
    assert np.array_equal(ctx.download(L.FIELD_V).reshape(-1, 3).view(np.uint32), marks)
    assert np.array_equal(ctx.download(L.FIELD_X).reshape(-1, 3), sc.x)
    ctx.close()


@pytest.mark.parametrize("n", [131070, 131072, 175000])
def test_fields_in_pieces(n):
    """Pieces of 43,690 particles through the halves of the staging memory."""
    sc = scenes.tiny_box(seed=2, fluid_counts=(3, 3, 3), cells=(120, 120, 120))
    rng = np.random.Generator(np.random.PCG64(n))
    x = scenes.lattice((0.1, 0.1, 0.1), (56, 56, 56)).astype(np.float32)
    sc.x = np.ascontiguousarray(x[rng.permutation(len(x))[:n]])
    sc.kind, sc.v = np.zeros(n, np.int32), np.zeros((n, 3), np.float32)
    ctx = L.Context(sc.params, sc.n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    assert np.array_equal(ctx.download(L.FIELD_X).reshape(-1, 3), sc.x)
    for k in (1, 3):
        marks = (k * np.arange(3 * n, dtype=np.uint32) * 2654435761 & 0x7FFFFFFF).reshape(-1, 3)
        ctx.upload_field(L.FIELD_V, marks.view(np.float32))
        assert np.array_equal(ctx.download(L.FIELD_V).reshape(-1, 3).view(np.uint32), marks)
    assert np.array_equal(ctx.download(L.FIELD_X).reshape(-1, 3), sc.x)
    ctx.close()
