"""Field output copied by several threads: arrays just below and above the size
where the copy is shared out (8 MB), and above the one where its chunks grow
(32 MB), none a whole number of chunks.  In an elastic analysis every voxel
holds sigma = C(phase) : eps (tensor shear); the bar is 1e-9 of the largest
stress, FP64 rounding of six products with room for the fields' own update."""
import numpy as np
import pytest

import mat3d_amd as m

pytestmark = pytest.mark.gpu

MAT = np.array([[350e9, 0.22, np.inf, 0, 1, 0, 0], [70e9, 0.32, np.inf, 0, 1, 0, 0]])


def stiffness(E, nu):
    la, mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
    C = np.zeros((6, 6))
    C[:3, :3] = la
    C[range(3), range(3)] += 2 * mu
    C[range(3, 6), range(3, 6)] = 2 * mu
    return C


@pytest.mark.parametrize("behav", ["e", "ep"])
@pytest.mark.parametrize("shape", [(55, 56, 56), (56, 56, 56), (65, 63, 45), (104, 104, 98)])
def test_fields_of_large_grids(shape, behav):
    ids = (np.random.default_rng(2).uniform(size=shape) > 0.4).astype(np.int32)
    s = m.FFT_Analysis3D(*shape, behav, precision="fp64")
    s.material(MAT, ids)
    E = np.array([1e-3, -2e-4, 3e-4, 2e-4, 0, 1e-4])
    s.setLoad(E, np.eye(6)[0])
    s.runAnalysis(1e-2, 1e-2, 1)
    # "ep" exports the next increment's start: after one increment twice the strain
    scale = 0.5 if behav == "ep" else 1.0
    for _ in range(2):  # the second call finds the buffers there
        eps, sig = s.fields()
        eps, sig = eps.reshape(-1, 6), sig.reshape(-1, 6)
        for k in (0, 1):
            of = ids.reshape(-1) == k
            ref = scale * eps[of] @ stiffness(*MAT[k, :2]).T
            assert np.abs(sig[of] - ref).max() < 1e-9 * np.abs(ref).max()
