"""Field and state output of at least 8 MB into every kind of memory that a C
caller may pass: pageable (copied by several threads), pinned and device
memory (the transfer's own target), from the start of the allocation and from
inside it.  The same bits everywhere, and nothing written beyond the array."""
import ctypes as ct

import numpy as np
import pytest
import torch

import mat3d_amd as m

pytestmark = pytest.mark.gpu

MAT = np.array([[350e9, 0.22, np.inf, 0, 1, 0, 0], [70e9, 0.32, np.inf, 0, 1, 0, 0]])


def targets(n, offset):
    """name, whole tensor of n + 2 * offset values, view of the n in the middle"""
    for name, kw in (("pageable", {}), ("pinned", {"pin_memory": True}), ("device", {"device": "cuda:0"})):
        t = torch.full((n + 2 * offset,), -7.0, dtype=torch.float64, **kw)
        yield name, t, t[offset : offset + n]


def call(f, h, lc, views):
    torch.cuda.synchronize()
    p = [ct.cast(v.data_ptr(), ct.POINTER(ct.c_double)) for v in views]
    assert f(h, *lc, *p) == 0


@pytest.mark.parametrize("offset", [0, 3])
@pytest.mark.parametrize("shape,behav", [((56, 56, 56), "e"), ((104, 104, 98), "ep")])
def test_kinds_of_memory(shape, behav, offset):
    ids = (np.random.default_rng(2).uniform(size=shape) > 0.4).astype(np.int32)
    s = m.FFT_Analysis3D(*shape, behav, precision="fp64")
    s.material(MAT, ids)
    s.setLoad(np.array([1e-3, -2e-4, 3e-4, 2e-4, 0, 1e-4]), np.eye(6)[0])
    s.runAnalysis(1e-2, 1e-2, 1)
    N = int(np.prod(shape))
    calls = [(m.lib().m3d_elastic_get_fields, (0,), 6 * N, s.fields())]
    if behav == "ep":
        calls.append((m.lib().m3d_elastic_get_state, (), N, s.history()))
    for f, lc, n, ref in calls:
        for (name, a, va), (_, b, vb) in zip(targets(n, offset), targets(n, offset)):
            call(f, s._h, lc, (va, vb))
            for t, v, r in ((a, va, ref[0]), (b, vb, ref[1])):
                assert (v.cpu().numpy() == np.asarray(r).reshape(-1)).all(), name
                rest = torch.cat([t[:offset], t[offset + n :]]).cpu()
                assert (rest == -7.0).all(), name
    s.close()
