"""nn_neighbors_noalloc with 16 and 4 lanes per particle against the FP32
oracle's lists: particle counts around a lane group, a wavefront and the limit
between the two forms, particles in random order, a row length that is not a
multiple of a group, and the grid's faces."""
import ctypes

import numpy as np
import pytest
import torch

from nonnewton_amd import _lib as L
from nonnewton_amd import scenes
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cap", [(1, 60), (4, 61), (17, 60), (65, 67), (131072, 60), (131073, 61)])
def test_lists_equal_the_oracles(n, cap):
    side = 52 if n > 1000 else 6
    sc = scenes.tiny_box(seed=1, fluid_counts=(3, 3, 3), cells=(2 * side, 2 * side, 2 * side))
    rng = np.random.Generator(np.random.PCG64(n))
    x = scenes.lattice((0.0, 0.0, 0.0), (side, side, side)).astype(np.float32)
    x = x + rng.uniform(0.0, 0.004, x.shape).astype(np.float32)
    sc.x = np.ascontiguousarray(x[rng.permutation(len(x))[:n]])
    sc.kind, sc.v = np.zeros(n, np.int32), np.zeros((n, 3), np.float32)
    o = O.OracleSim.from_scene(sc, precision="f32")
    o.init()
    on, oc = o.neighbors()
    xt = torch.from_numpy(sc.x).cuda()
    nbr = torch.full((n, cap), 7, dtype=torch.int32, device="cuda")
    cnt, status = torch.full((n,), 7, dtype=torch.int32, device="cuda"), torch.full((1,), 7, dtype=torch.int32, device="cuda")
    p = L.params_struct(sc.params)
    L.check(L.load().nn_neighbors_noalloc(ctypes.byref(p), xt.data_ptr(), n, nbr.data_ptr(), cnt.data_ptr(), cap,
                                          status.data_ptr(), torch.cuda.current_stream().cuda_stream), "noalloc")
    assert int(status.cpu()[0]) == 0
    assert np.array_equal(cnt.cpu().numpy(), oc)
    got = nbr.cpu().numpy()
    assert np.array_equal(got[:, : on.shape[1]], on)
    assert np.all(got[:, on.shape[1]:] == -1)
