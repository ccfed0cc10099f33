"""Copies to the host: a grid and a species read back equal what was uploaded,
at sizes on both sides of the staging rules (192 KiB, 1 MiB, odd numbers of
512 KiB pieces), into memory that was never touched and into memory in use."""
import ctypes
import mmap

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,nz", [(5, 31), (157, 157), (129, 1017), (257, 2047), (700, 1501)])
def test_grid_download(nr, nz):
    from pdp3_amd import capi

    d = 5e-4
    sim = capi.Simulation(nr, nz, (nr - 1) * d, (nz - 1) * d, 0.5 * d / 3e8)
    a = np.random.default_rng(nr).standard_normal((nr, nz))
    sim.set_field("E_phi", a)
    dbl = ctypes.POINTER(ctypes.c_double)
    with mmap.mmap(-1, a.nbytes + 4096) as fresh:  # not one page of it touched
        view = np.frombuffer(fresh, np.float64, a.size, offset=8 * 3)
        assert sim.L.pdp3_grid_download(sim.h, 1, view.ctypes.data_as(dbl)) == 0
        assert np.array_equal(view.reshape(a.shape), a)
        del view
    used = np.full((nr, nz), 7.0)
    assert sim.L.pdp3_grid_download(sim.h, 1, used.ctypes.data_as(dbl)) == 0
    assert np.array_equal(used, a)
    assert np.array_equal(sim.field("E_phi"), a)
    sim.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_species_download(precision):
    from pdp3_amd import capi

    rng = np.random.default_rng(5)
    n, d = 300007, 5e-4
    sim = capi.Simulation(65, 257, 64 * d, 256 * d, 0.5 * d / 3e8, precision=precision)
    r, z = d / 2 + rng.random(n) * 63 * d, d / 2 + rng.random(n) * 255 * d
    v = rng.normal(0, 1e6, (3, n))
    alive = (rng.random(n) > 0.2).astype(np.uint8)
    sim.add_plasma(-1, 1.0, r, z, v[0], v[1], v[2], np.arange(n, dtype=float), alive)
    out = sim.download(0)
    tol = 0.0 if precision == 0 else 1e-6
    for k, x in (("r", r), ("z", z), ("vr", v[0]), ("vphi", v[1]), ("vz", v[2]), ("w", np.arange(n, dtype=float))):
        assert np.max(np.abs(out[k] - x)) <= tol * np.max(np.abs(x)), k
    assert np.array_equal(out["alive"], alive)
    sim.close()
