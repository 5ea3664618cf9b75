"""Particle fields back on the host (GPU): every field of a state uploaded and
read back is the value uploaded, rounded once to the kernel precision (no
tolerance), for one particle, for counts around a workgroup, for arrays larger
than a chunk of the read-back (32 MB), for fewer rows than there are particles
and for fields that are not held (all zeros)."""
import ctypes as C

import numpy as np
import pytest

import ftrack
import mpmw
import workloads

pytestmark = pytest.mark.gpu


def rounded(a, prec, exact):
    a = np.asarray(a)
    return a if exact or prec == "fp64" or a.dtype != np.float64 else a.astype(np.float32).astype(np.float64)


def workpiece_state(n, rng, back):
    d = mpmw.make_arrays(n)
    for k, v in d.items():
        if v.dtype == np.float64:
            v[...] = rng.uniform(0.5, 2.0, v.shape)
    d["pos"][...] = rng.uniform(0, 2e-3, (n, 3))
    d["mass"][:], d["volume"][:] = 1.25, 0.75
    d["id"][:] = rng.permutation(n)
    d["status"][:] = rng.integers(0, 5, n)
    d["fext"][...] = 0.0
    if not back:
        d["backstress"][...] = 0.0
    return d


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("n,back", [(1, True), (255, False), (257, True), (800_003, False)])
def test_workpiece_state_comes_back(n, back, prec):
    d = workpiece_state(n, np.random.default_rng(n), back)
    s = mpmw.Solver(**workloads.params_dict(precision=mpmw.FP64 if prec == "fp64" else mpmw.FP32))
    s.set_particles(d)
    g = s.get_particles()
    for k, v in d.items():
        assert np.array_equal(g[k], rounded(v, prec, k == "pos")), k
    # the first rows only, and only some arrays, into memory that held other values
    m = max(1, n // 3)
    pos, fext, ids = np.full((m, 3), 7.0), np.full((m, 3), 7.0), np.full(m, 7, np.int32)
    a = mpmw.ParticleArrays()
    a.n = m
    a.pos, a.fext, a.id = mpmw._p(pos), mpmw._p(fext), mpmw._p(ids, C.POINTER(C.c_int32))
    assert mpmw.lib().mpmw_get_particles(s.h, C.byref(a)) == 0 and a.n == m
    assert np.array_equal(pos, d["pos"][:m]) and not fext.any() and np.array_equal(ids, d["id"][:m])
    s.close()


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("n", [1, 256, 600_001])
def test_ftrack_state_comes_back(n, prec):
    rng = np.random.default_rng(n)
    d = ftrack.make_arrays(n)
    for k, v in d.items():
        if v.dtype == np.float64:
            v[...] = rng.uniform(0.5, 2.0, v.shape)
    d["pos"][...] = rng.uniform(0, 2e-3, (n, 3))
    for k in ("F", "Fp"):   # held as their difference from the identity: values whose difference is exact
        d[k][...] = np.eye(3).reshape(9) + rng.integers(-64, 64, (n, 9)) / 1024.0
    d["id"][:], d["status"][:], d["lod"][:] = rng.permutation(n), rng.integers(0, 5, n), rng.integers(0, 3, n)
    s = ftrack.Solver(ftrack.default_params(precision=ftrack.FP64 if prec == "fp64" else ftrack.FP32))
    s.set_particles(d)
    g = s.get_particles()
    for k, v in d.items():
        assert np.array_equal(g[k], rounded(v, prec, k == "pos")), k
    some = s.get_particles(fields=("F", "lod"))
    assert set(some) == {"F", "lod", "id", "status"} and np.array_equal(some["F"], d["F"])
    s.close()
