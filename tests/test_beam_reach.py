"""The box of cells beyond which a launch's patches skip the heat sources:
against the test of every cell on the host, and on the device on meshes of
which a beam reaches a small part."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from adamantine_amd.problem import (SOURCE_CUBE, SOURCE_ELECTRON_BEAM,
                                    SOURCE_GOLDAK, BeamState)

SRC = os.path.join(os.path.dirname(__file__), "cxx", "beam_reach.cpp")
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("reach") / "beam_reach.so")
    # -no-hip-rt: without the HIP runtime, of which a process must not load a
    # second one beside torch's
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-x",
                    "hip", "--offload-arch=gfx950", "--cuda-host-only", "-O2",
                    "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared",
                    "-no-hip-rt", "-I", os.path.join(ROOT, "include"), "-o",
                    out, SRC], check=True)
    L = C.CDLL(out)
    L.missed_cells.restype = C.c_int64
    return L


def rotation(rng):
    q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    return q


def random_beam(rng, origin, extent, h):
    s = BeamState()
    s.type = int(rng.choice([SOURCE_GOLDAK, SOURCE_ELECTRON_BEAM,
                             SOURCE_CUBE]))
    s.on = int(rng.rand() < 0.8)
    # inside the mesh, out of it, and on cell faces
    c = origin + rng.uniform(-0.5, 1.5, 3) * extent
    if rng.rand() < 0.3:
        c = origin + np.rint((c - origin) / h) * h
    s.center[:] = c
    r = 10.0 ** rng.uniform(-2, 0.5) * extent.min()
    s.radius_squared = r * r
    s.depth = 10.0 ** rng.uniform(-2, 0.5) * extent[2]
    lo, hi = np.sort([c, c + rng.uniform(-0.3, 0.3, 3) * extent], axis=0)
    s.cube_min[:], s.cube_max[:] = lo, hi
    if s.type != SOURCE_CUBE and rng.rand() < 0.2:
        s.rotated = 1
        s.rotation[:] = rotation(rng).ravel()
    return s


def missed(lib, beams, origin, h, nc):
    arr = (BeamState * max(1, len(beams)))(*beams)
    outside = C.c_int64()
    dp = C.POINTER(C.c_double)
    nc = np.array(nc, np.int32)
    n = lib.missed_cells(arr, len(beams), origin.ctypes.data_as(dp),
                         h.ctypes.data_as(dp),
                         nc.ctypes.data_as(C.POINTER(C.c_int32)),
                         C.byref(outside))
    return n, outside.value


def test_reach_misses_no_cell(lib):
    rng = np.random.RandomState(4)
    total = 0
    for k in range(600):
        nc = rng.randint(1, 24, 3)
        h = 10.0 ** rng.uniform(-5, 0) * rng.uniform(0.3, 1.0, 3)
        origin = rng.choice([0.0, -1.0, 5.0]) * h * nc
        beams = [random_beam(rng, origin, h * nc, h)
                 for _ in range(rng.randint(0, 5))]
        n, outside = missed(lib, beams, origin, h, nc)
        assert n == 0, k
        total += outside
    assert total > 100000  # the box does leave cells out


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("what", ["center", "radius", "depth", "cube"])
def test_reach_not_finite(lib, bad, what):
    rng = np.random.RandomState(6)
    nc, h, origin = np.array([9, 7, 5]), np.full(3, 0.1), np.zeros(3)
    for k in range(20):
        s = random_beam(rng, origin, h * nc, h)
        if what == "center":
            s.center[k % 3] = bad
        elif what == "radius":
            s.radius_squared = bad
        elif what == "depth":
            s.depth = bad
        else:
            s.cube_min[k % 3] = bad
        assert missed(lib, [s], origin, h, nc)[0] == 0, k


def problem(degree, kind, place):
    """A mesh of many patches and a small source at one of its places."""
    from adamantine_amd.problem import Beam
    from adamantine_amd.workloads import plain_large
    cells = {1: (40, 22, 6), 2: (36, 17, 6), 3: (22, 14, 5)}[degree]
    p = plain_large(n_cells=cells)
    p.fe_degree = degree
    x, y, z = p.extent
    at = {"corner": (0.02 * x, 0.03 * y, z), "middle": (0.47 * x, 0.52 * y, z),
          "edge": (x, 0.4 * y, z), "inside": (0.7 * x, 0.2 * y, 0.5 * z),
          "beside": (-0.01 * x, 0.6 * y, z)}[place]
    if kind == SOURCE_CUBE:
        w = 0.04 * x
        p.beams = [Beam(type=kind, start_time=0.0, end_time=1.0, value=1e15,
                        min_point=tuple(c - w for c in at),
                        max_point=tuple(c + w for c in at))]
    else:
        b = p.beams[0]
        b.type, b.radius, b.depth = kind, 60e-6, 90e-6
        b.segments = [(1e-9, 0.0, at), (1.0, 1.0, at)]
    return p


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [SOURCE_GOLDAK, SOURCE_ELECTRON_BEAM,
                                  SOURCE_CUBE])
@pytest.mark.parametrize("place", ["corner", "middle", "edge", "inside",
                                   "beside"])
@pytest.mark.parametrize("degree", [1, 2, 3])
def test_small_source(degree, place, kind):
    """At 300 K everywhere the result is the source (and rounding): a cell
    left out shows at its full size."""
    import torch
    from adamantine_amd.thermal import ThermalOperatorDevice
    from oracle.oracle import Oracle
    p = problem(degree, kind, place)
    op, o = ThermalOperatorDevice(p), Oracle(p)
    T = np.full(p.n_dofs, 300.0)
    for obj in (op, o):
        obj.set_time(0.1)
    want = o.vmult(T)
    dst = op.initialize_dof_vector(7.0)
    op.vmult(dst, torch.tensor(T, device="cuda"))
    got = dst.cpu().numpy()
    peak = np.abs(want).max()
    assert 0 < np.count_nonzero(np.abs(want) > 1e-6 * peak) < 0.2 * p.n_dofs
    # rounding of the source's values (an exponential, ~1e2 operations), and
    # of the stiffness of the constant field
    assert np.abs(got - want).max() <= 1e-12 * peak
