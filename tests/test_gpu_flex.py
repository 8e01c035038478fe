"""The passes for line lengths without a compile-time kernel (m3d_flex.hpp,
m3d_flex_basic.hip) against the FP64 oracle: every radix 2..16, one to four
passes per line, ragged last tiles, odd rows per z tile (thermal transforms
rows in pairs), and the 1024-thread forms of long lines.  Bars as in
test_gpu_parity.py: same iteration counts and 1e-9 relative in FP64, C_eff
within 1e-6 in FP32 + polish."""
import numpy as np
import pytest

import mat3d_amd as m
import oracle
from mat3d_amd import gen

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b))


def field_rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def blocks(shape, seed):
    """Two phases in blocks of 2 voxels, about 30% phase 0."""
    half = tuple((v + 1) // 2 for v in shape)
    ids = (np.random.default_rng(seed).uniform(size=half) > 0.3).astype(np.int32)
    ids = ids.repeat(2, 0).repeat(2, 1).repeat(2, 2)[: shape[0], : shape[1], : shape[2]].copy()
    ids.reshape(-1)[:2] = [0, 1]
    return ids


MAT = np.array([[350e9, 0.22, np.inf, 0, 1, 0, 0], [70e9, 0.32, np.inf, 0, 1, 0, 0]])

# (x, y, z) line lengths; the last four: lines of more than 341 (x), 341 (y)
# and 682 (z) points, and of 7^3 and 13^2 points
ELASTIC = [(4, 3, 5), (13, 11, 7), (14, 22, 15), (9, 25, 27), (10, 26, 12), (45, 10, 49), (33, 6, 98), (343, 2, 6),
           (4, 350, 10), (3, 4, 700), (169, 5, 8)]


@pytest.mark.parametrize("shape", ELASTIC)
def test_elastic_lines(shape):
    ids = blocks(shape, 3)
    for mat in (MAT, MAT[::-1].copy()):  # stress and strain base
        o = oracle.Elastic(*shape, "e")
        o.material(mat, ids)
        r = o.homogenization(1e-6, 1e-6)
        s = m.FFT_Analysis3D(*shape, "e", precision="fp64")
        s.material(mat, ids)
        s.homogenization(1e-6, 1e-6)
        assert [i["iterations"] for i in s.info] == r["iters"]
        assert rel(s.CHomo, r["C"]) < 1e-9
        eps_o, sig_o = o.fields()
        eps, sig = s.fields(5)
        assert field_rel(sig, sig_o) < 1e-9 and field_rel(eps, eps_o) < 1e-9
    p = m.FFT_Analysis3D(*shape, "e", precision="fp32_polish")
    p.material(mat, ids)
    p.homogenization(1e-6, 1e-6)
    assert rel(p.CHomo, r["C"]) < 1e-6


# Nx <= Ny (the flux base folds x with Ny); the last two: lines of more than
# 682 points
THERMAL = [(3, 5, 7), (4, 4, 5), (14, 15, 26), (22, 25, 33), (9, 49, 10), (5, 686, 4), (3, 4, 1400)]


@pytest.mark.parametrize("shape", THERMAL)
def test_thermal_lines(shape):
    ids = blocks(shape, 5)
    for km, ki in ((1.0, 12.0), (12.0, 1.0)):  # gradient and flux base
        o = oracle.Thermal(*shape)
        o.material(km, ki, ids)
        r = o.homogenization(1e-6, 1e-6)
        s = m.FFT_analysis3d_thermal(*shape, precision="fp64")
        s.material(km, ki, ids)
        s.homogenization(1e-6, 1e-6)
        assert [i["iterations"] for i in s.info] == r["iters"]
        assert rel(s.KHomo, r["K"]) < 1e-9
        g_o, q_o = o.fields()
        g, q = s.fields(2)
        assert field_rel(g, g_o) < 1e-9 and field_rel(q, q_o) < 1e-9
        p = m.FFT_analysis3d_thermal(*shape, precision="fp32_polish")
        p.material(km, ki, ids)
        p.homogenization(1e-6, 1e-6)
        assert rel(p.KHomo, r["K"]) < 1e-6


MAT_J2 = np.array([[400e9, 0.20, np.inf, 0, 1, 0, 0], [70e9, 0.30, 100e6, 1e9, 1, 0, 0]])
MAT_J2N = np.array([[400e9, 0.20, np.inf, 0, 1, 0, 0], [70e9, 0.30, 100e6, 1e9, 0.5, 0, 0]])
MAT_ED = np.array([[400e9, 0.20, np.inf, 0, 1, 1e-3, 2e3], [70e9, 0.30, np.inf, 0, 1, 1e-3, 8e2]])


# the last three: lines of more than 170 (x, start stage), 256 (x) and 512
# (z) points
@pytest.mark.parametrize("shape", [(4, 3, 5), (10, 13, 15), (12, 9, 22), (175, 3, 4), (273, 2, 5), (3, 4, 520)])
@pytest.mark.parametrize("behav,mat,strain", [("ep", MAT_J2, 0.004), ("ep", MAT_J2N, 0.004), ("ed", MAT_ED, 0.0018)])
def test_load_path_lines(shape, behav, mat, strain):
    ids = blocks(shape, 7)
    X0 = np.eye(6)[1]
    o = oracle.Elastic(*shape, behav)
    o.material(mat, ids)
    o.set_load(strain * X0, X0)
    it = o.run(1e-6, 1e-6, 3)
    s = m.FFT_Analysis3D(*shape, behav, precision="fp64")
    s.material(mat, ids)
    s.setLoad(strain * X0, X0)
    info = s.runAnalysis(1e-6, 1e-6, 3)
    assert info["iters_fp64"] == it
    P, P_o = s.prop_homogenized, o.prop_homogenized()
    eps, sig = s.fields()
    eps_o, sig_o = o.fields()
    assert field_rel(P, P_o) < 1e-9
    assert field_rel(sig, sig_o) < 1e-9 and field_rel(eps, eps_o) < 1e-9
    a, b = s.history()
    if behav == "ep":
        ep_o, se_o = o.j2_state()
        assert field_rel(a, ep_o) < 1e-9 and field_rel(b, se_o) < 1e-9
    else:
        assert np.abs(a - o.damage_state()).max() < 1e-9


def test_line_limits():
    """What no workgroup's tile holds, and prime factors above 13, stay refused."""
    for shape in [(17, 8, 8), (8, 8, 34), (8, 704, 8), (704, 8, 8), (8, 8, 1372), (8, 8, 693)]:
        with pytest.raises(m.M3DError) as e:
            m.FFT_Analysis3D(*shape, "e")
        assert e.value.code == -2, shape
