"""Kinetic-energy, trigger and pair sums around the grid size up to which
kernels finish their own sums (32 blocks: 16,384 free atoms of one mass, 8,192
of two masses or bodies), with energies switched on and off between kicks."""
import numpy as np
import pytest

import bench
from emdee_amd.water_box import KB, water_system

pytestmark = pytest.mark.gpu


def run(lib, md, dt, compute):
    rec = []
    for on in compute:
        md.Options.Compute = on
        lib.boost(md, 1.0, 0.0, 0.5 * dt)
        lib.displace(md, 1.0, 0.0, dt)
        lib.boost(md, 1.0, 0.0, 0.5 * dt)
        rec.append([md.Energy.Potential, md.Virial, md.Kinetic.Total, md.Builds])
    return np.array(rec)


@pytest.mark.parametrize("natoms,masses", [(500, 1), (16384, 1), (16385, 1), (8192, 2), (8193, 2)])
def test_free_atoms(gpu, oracle, natoms, masses):
    R, L = bench.fcc_lattice(natoms, 0.8442)
    R = R + 0.05 * np.random.default_rng(5).standard_normal(R.shape)
    types = 1 + np.arange(natoms, dtype=np.int32) % masses
    out = []
    for lib in (gpu, oracle):
        md = lib.system(1, 1, 2.5, 0.3, natoms, types, np.array([1.0, 2.0][:masses]), None)
        for t in range(1, masses + 1):
            lib.EmDee_set_pair_model(md, t, t, lib.EmDee_pair_lj_cut(1.0, 1.0), 0.0)
        lib.upload(md, "box", np.array([L]))
        lib.upload(md, "coordinates", R)
        lib.random_momenta(md, 1.0, True, 11)
        out.append(run(lib, md, 0.005, [True, False, True, True, False, False, True] * 2))
    # sums of 5e5 terms of either sign: 1e-16 sqrt(5e5) on sums a tenth of their terms, grown twofold over 14 steps
    np.testing.assert_allclose(out[0], out[1], rtol=2e-11)


@pytest.mark.parametrize("nmol", [300, 8192, 8193])
def test_bodies(gpu, oracle, nmol):
    out = []
    for lib in (gpu, oracle):
        md, _ = water_system(lib, nmol, 3, rc=6.0, skin=1.0, coul="damped", alpha=0.3)
        lib.random_momenta(md, KB * 298.0, True, 11)
        out.append(run(lib, md, 1.0, [True, False, True, True]))
    np.testing.assert_allclose(out[0], out[1], rtol=1e-9)   # principal axes good to 1e-10 (test_gpu_rigid)
