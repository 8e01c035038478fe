"""The kz tiles of the x and y passes along lines of 32 and 48 points against
the FP64 oracle: grids whose Nz/2+1 is smaller than a tile, a whole number of
tiles, and one or two kz more than that (FP32 tiles 17 and 13, FP64 tiles 8 and 5).
Bars as in test_gpu_parity.py: same iteration counts and 1e-9 relative in FP64,
C_eff within 1e-6 in FP32 + polish."""
import numpy as np
import pytest

import mat3d_amd as m
import oracle

pytestmark = pytest.mark.gpu

MAT = np.array([[350e9, 0.22, np.inf, 0, 1, 0, 0], [70e9, 0.32, np.inf, 0, 1, 0, 0]])


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b))


# (x, y, z); Nz/2+1 = 3, 8, 9, 13, 14, 19, 26
@pytest.mark.parametrize("shape", [(32, 48, 4), (48, 32, 14), (32, 32, 16), (48, 48, 24), (32, 48, 26), (32, 32, 36),
                                   (48, 48, 50)])
def test_short_lines(shape):
    ids = (np.random.default_rng(5).uniform(size=shape) > 0.3).astype(np.int32)
    o = oracle.Elastic(*shape, "e")
    o.material(MAT, ids)
    r = o.homogenization(1e-6, 1e-6)
    s = m.FFT_Analysis3D(*shape, "e", precision="fp64")
    s.material(MAT, ids)
    s.homogenization(1e-6, 1e-6)
    assert [i["iterations"] for i in s.info] == r["iters"]
    assert rel(s.CHomo, r["C"]) < 1e-9
    p = m.FFT_Analysis3D(*shape, "e", precision="fp32_polish")
    p.material(MAT, ids)
    p.homogenization(1e-6, 1e-6)
    assert rel(p.CHomo, r["C"]) < 1e-6


MAT_J2 = np.array([[400e9, 0.20, np.inf, 0, 1, 0, 0], [70e9, 0.30, 100e6, 1e9, 1, 0, 0]])


@pytest.mark.parametrize("n", [32, 48, 96, 128, 192])
def test_basic_x_tiles(n):
    """J2 load path over 17 kz: x tiles of 8, 5, 2 and 2 kz on 256 threads (32,
    48, 96, 128 points) and of 2 on 512 (192), the last one ragged."""
    j2_path((n, 32, 32))


# planes * (Nz/2+1) / 384: x tiles of 2, 11 and 1 kz, y tiles of 1, 1 and 6
@pytest.mark.parametrize("shape", [(20, 40, 44), (10, 90, 98), (100, 10, 50)])
def test_basic_tiles_without_compile_time_kernels(shape):
    j2_path(shape)


def j2_path(shape):
    ids = (np.random.default_rng(7).uniform(size=shape) > 0.3).astype(np.int32)
    X0 = np.eye(6)[1]
    o = oracle.Elastic(*shape, "ep")
    o.material(MAT_J2, ids)
    o.set_load(0.002 * X0, X0)
    it = o.run(1e-6, 1e-6, 2)
    s = m.FFT_Analysis3D(*shape, "ep", precision="fp64")
    s.material(MAT_J2, ids)
    s.setLoad(0.002 * X0, X0)
    assert s.runAnalysis(1e-6, 1e-6, 2)["iters_fp64"] == it
    P, P_o = s.prop_homogenized, o.prop_homogenized()
    assert np.abs(P - P_o).max() < 1e-9 * np.abs(P_o).max()
    for a, b in zip(s.fields(), o.fields()):
        assert np.abs(a - b).max() < 1e-9 * np.abs(b).max()
