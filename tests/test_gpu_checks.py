"""When the equilibrium-check passes are launched does not change a solve.  A
solve that needs a check which its launched iteration does not hold waits and
goes on from the same iterate: with a wide tolerance the first check is needed
in iteration 2, before the host has read any state, so every solve waits
there.  Iterations and tensors against the FP64 oracle (1e-9 relative, as in
the parity tests).  The option "chunk" once grouped iterations: every value
that it takes gives the same bits, in the same time."""
import time

import numpy as np
import pytest

import mat3d_amd as m
import oracle
from mat3d_amd import gen

pytestmark = pytest.mark.gpu
CHUNKS = [0, 1, 3, 7]


def solve(shape, ids, precision, tol, chunk):
    s = m.FFT_Analysis3D(*shape, "e", precision=precision)
    s.set_option("chunk", chunk)
    s.material(gen.MAT_C2, ids)
    s.homogenization(tol, tol)
    out = s.CHomo.copy(), [(i["iterations"], i["status"], i["eqVar"], i["diff_sum"], i["diff_eq"]) for i in s.info]
    s.close()
    return out


# compile-time and run-time line lengths
@pytest.mark.parametrize("shape", [(32, 32, 32), (20, 24, 18)])
@pytest.mark.parametrize("tol", [0.3, 1e-2, 1e-6])
def test_fp64_solves(shape, tol):
    n = max(shape)
    ids = gen.fibres(n, 3, 0.3, seed=2, length=n // 2)[: shape[0], : shape[1], : shape[2]].copy()
    o = oracle.Elastic(*shape, "e")
    o.material(gen.MAT_C2, ids)
    ref = o.homogenization(tol, tol)
    first = solve(shape, ids, "fp64", tol, CHUNKS[0])
    assert [i[0] for i in first[1]] == list(ref["iters"])
    assert np.linalg.norm(first[0] - ref["C"]) < 1e-9 * np.linalg.norm(ref["C"])
    for chunk in CHUNKS[1:]:
        C, info = solve(shape, ids, "fp64", tol, chunk)
        assert info == first[1] and (C == first[0]).all()


@pytest.mark.parametrize("shape", [(32, 32, 32), (20, 24, 18)])
@pytest.mark.parametrize("tol", [1e-2, 1e-6])
def test_fp32_polish(shape, tol):
    n = max(shape)
    ids = gen.fibres(n, 3, 0.3, seed=2, length=n // 2)[: shape[0], : shape[1], : shape[2]].copy()
    first = solve(shape, ids, "fp32_polish", tol, CHUNKS[0])
    for chunk in CHUNKS[1:]:
        C, info = solve(shape, ids, "fp32_polish", tol, chunk)
        assert info == first[1] and (C == first[0]).all()


@pytest.mark.parametrize("precision", ["fp64", "fp32_polish"])
def test_chunk_costs_nothing(precision):
    ids = gen.fibres(32, 3, 0.3, seed=2, length=16)
    best = {}
    for chunk in (0, 200):
        s = m.FFT_Analysis3D(32, 32, 32, "e", precision=precision)
        s.set_option("chunk", chunk)
        s.material(gen.MAT_C2, ids)
        times = []
        for _ in range(6):
            t = time.perf_counter()
            s.homogenization(1e-6, 1e-6)
            times.append(time.perf_counter() - t)
        best[chunk] = min(times)
        s.close()
    # idle groups of 200 iterations took 5 to 10 times as long
    assert best[200] < 3 * best[0], best


@pytest.mark.parametrize("precision", ["fp64", "fp32_polish"])
def test_batch_of_solves_that_stop_apart(precision):
    # six load cases of four structures of other contrast, two grid shapes
    res = []
    for chunk in CHUNKS:
        b = m.Batch(precision=precision)
        b.set_option("chunk", chunk)
        for k, n in enumerate((24, 24, 30, 24, 30)):
            mat = gen.MAT_C2.copy()
            mat[0, 0] *= 2.0 ** k
            b.add(mat, gen.spheres(n, 3, 0.1 + 0.04 * k, seed=k))
        b.homogenization(1e-6, 1e-6)
        r = [b.result(k) for k in range(5)]
        res.append([(x["CHomo"].tolist(), [(i["iterations"], i["eqVar"]) for i in x["info"]]) for x in r])
        b.close()
    assert len({i[0] for x in res[0] for i in x[1]}) > 1
    for r in res[1:]:
        assert r == res[0]
