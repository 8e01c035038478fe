"""setLoad of FFT_Analysis2D has filled the strain when it returns: fields()
right after it gives the load at every point, on a new handle and after a
run, at the smallest and the largest plate."""
import numpy as np
import pytest

import mat3d_amd as m

pytestmark = pytest.mark.gpu

Q = [68.9e9, 0.35, 400e9, 0.23]


@pytest.mark.parametrize("n", [32, 512])
def test_fields_right_after_set_load(n):
    rve = (np.random.default_rng(n).uniform(size=n * n) > 0.25).astype(np.float64)
    E1, E2 = np.array([0.002, 0.001j, 0.003]), np.array([-0.004, 0.005, 0.006 + 0.007j])
    g = m.FFT_Analysis2D(n, n)
    g.material(Q, rve)
    g.setLoad(E1)
    eps, sig = g.fields()
    assert (eps == E1).all() and (sig == 0).all()
    g.runAnalysis()
    _, run_sig = g.fields()
    for E in (E2, E1):
        g.setLoad(E)
        eps, sig = g.fields()
        assert (eps == E).all()
        # the stress is the last run's until the next one
        assert (sig == run_sig).all()
