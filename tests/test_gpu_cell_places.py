"""Particles' places in their cells, members read eight at a time: cells of 1,
7, 8, 9, 16, 17, 48, 49 and 50 particles in random order, by the context's search
and by nn_neighbors_noalloc, against the FP32 oracle's lists."""
import ctypes

import numpy as np
import pytest
import torch

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [1, 2])
def test_members_of_a_cell(seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    sc = scenes.tiny_box(seed=seed, fluid_counts=(3, 3, 3), cells=(40, 40, 40))
    h = 2.0 * 2.0 * sc.params.particle_radius
    parts = []
    for c, members in enumerate((1, 7, 8, 9, 16, 17, 48, 49, 50)):
        cell = np.array([1 + 3 * (c % 3), 1 + 3 * (c // 3), 4])
        parts.append((cell + 0.5 + rng.uniform(-0.45, 0.45, (members, 3))) * h)
    x = np.concatenate(parts).astype(np.float32)
    sc.x = np.ascontiguousarray(x[rng.permutation(len(x))])
    n = len(sc.x)
    sc.kind, sc.v = np.zeros(n, np.int32), np.zeros((n, 3), np.float32)
    o = O.OracleSim.from_scene(sc, precision="f32")
    o.init()
    on, oc = o.neighbors()
    assert oc.max() > 40
    ctx = L.Context(sc.params, n)
    ctx.upload(sc.x, sc.kind, sc.v)
    ctx.init()
    nbr, cnt = ctx.neighbors()
    assert np.array_equal(cnt, oc) and np.array_equal(nbr[:, : on.shape[1]], on)
    ctx.close()
    xt = torch.from_numpy(sc.x).cuda()
    out = torch.full((n, 60), 7, dtype=torch.int32, device="cuda")
    num, status = torch.full((n,), 7, dtype=torch.int32, device="cuda"), torch.full((1,), 7, dtype=torch.int32, device="cuda")
    p = L.params_struct(sc.params)
    L.check(L.load().nn_neighbors_noalloc(ctypes.byref(p), xt.data_ptr(), n, out.data_ptr(), num.data_ptr(), 60,
                                          status.data_ptr(), torch.cuda.current_stream().cuda_stream), "noalloc")
    assert int(status.cpu()[0]) == 0
    assert np.array_equal(num.cpu().numpy(), oc) and np.array_equal(out.cpu().numpy()[:, : on.shape[1]], on)
