"""The row pass of FFT_Analysis2D (backward y FFT, strain, polarisation,
forward y FFT in one launch) at every y length, with its stored fields and
row sums, against the FP64 oracle; a second homogenization continues from the
fields of the first, as the reference does."""
import numpy as np
import pytest

import mat3d_amd as m
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nx,Ny", [(32, 32), (32, 48), (48, 64), (32, 96), (64, 128), (48, 192), (32, 256), (32, 512)])
def test_row_lengths(Nx, Ny):
    rng = np.random.default_rng(Ny)
    rve = (rng.uniform(size=Nx * Ny) > 0.25).astype(np.float64)
    q = [68.9e9, 0.35, 400e9, 0.23]
    o = oracle.Elastic2D(Nx, Ny)
    o.material(q, rve)
    o.set_load([0.002, 0.001j, 0.003])
    g = m.FFT_Analysis2D(Nx, Ny)
    g.material(q, rve)
    g.setLoad([0.002, 0.001j, 0.003])
    for _ in range(2):
        C_o, ep_o, sg_o = o.homogenization()
        C = g.homogenization()
        for a, b in ((C, C_o), (g.epHomo, ep_o), (g.sigHomo, sg_o)):
            assert np.abs(a - np.asarray(b).reshape(a.shape)).max() < 1e-11 * np.abs(b).max()
        for a, b in zip(g.fields(), o.fields()):
            assert np.abs(a - b).max() < 1e-11 * np.abs(b).max()
    g.setLoad([0.002, 0.001j, 0.003])
    o.set_load([0.002, 0.001j, 0.003])
    g.runAnalysis()
    o.run()
    for a, b in zip(g.fields(), o.fields()):
        assert np.abs(a - b).max() < 1e-11 * np.abs(b).max()
