"""An error that another HIP call of the thread has left behind does not fail the
field transfers and mesh reads that launch nothing of it."""
import ctypes

import numpy as np
import pytest

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes
from nonnewton_amd.surface import Surface

pytestmark = pytest.mark.gpu


def leave_error():
    assert ctypes.CDLL("libamdhip64.so").hipSetDevice(12345) != 0


def test_transfers_after_an_error_of_another_call():
    sc = scenes.tiny_box()
    ctx = L.Context(sc.params, sc.n)
    leave_error()
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    for field in (L.FIELD_X, L.FIELD_V, L.FIELD_ACCELERATION):
        leave_error()
        a = ctx.download(field)
    leave_error()
    ctx.upload_field(L.FIELD_V, np.ones_like(a))
    leave_error()
    assert (ctx.download(L.FIELD_V) == 1).all()
    ctx.step()
    pool = L.Pool(1 << 30)
    slot = pool.admit(sc.params, sc.x, sc.kind, sc.v)
    pool.tick()
    leave_error()
    x = pool.read(slot, L.FIELD_X)
    assert np.isfinite(x).all()
    pool.close()
    s = Surface(voxel_size=0.02, particle_radius=0.01, smooth_radius=0.04, normals=True)
    s.run_context(ctx)
    leave_error()
    assert len(s.mesh()[0]) > 0
    s.close()
    ctx.close()
