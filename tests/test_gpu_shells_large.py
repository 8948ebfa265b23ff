"""Shell-ordered lists of systems past 16,384 atoms, and lists without shells
where one lane walks an atom's list, against the oracle."""
import numpy as np
import pytest

import bench
from emdee_amd.water_box import KB, water_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nmol,rc", [(5462, 8.0), (22000, 6.0)])
def test_water(gpu, oracle, nmol, rc):
    out, F = [], []
    for lib in (gpu, oracle):
        md, _ = water_system(lib, nmol, 8, rc=rc, skin=2.0, coul="damped", alpha=0.3)
        lib.random_momenta(md, KB * 298.0, True, 5)
        rec = []
        for _ in range(8):
            lib.boost(md, 1.0, 0.0, 1.0)
            lib.displace(md, 1.0, 0.0, 2.0)
            lib.boost(md, 1.0, 0.0, 1.0)
            rec.append([md.Energy.Potential, md.Kinetic.Total, md.Builds])
        out.append(np.array(rec))
        F.append(lib.download(md, "forces", (3 * nmol, 3)))
    np.testing.assert_allclose(out[0], out[1], rtol=1e-8)   # principal axes good to 1e-10 (test_gpu_rigid)
    # ... times the slope of a contact (1e2 of the force per A), grown over 8 steps
    assert np.max(np.abs(F[0] - F[1])) <= 1e-6 * np.max(np.abs(F[1]))


# two types take the multi-lane kernels up to 65,536 atoms; short lists beyond, and one type past 131,072, one lane
@pytest.mark.parametrize("natoms,types,rc", [(65536, 2, 2.5), (66000, 2, 2.5), (66000, 2, 3.2), (131072, 1, 3.2)])
def test_atoms(gpu, oracle, natoms, types, rc):
    R, L = bench.fcc_lattice(natoms, 0.8442)
    R = R + 0.05 * np.random.default_rng(5).standard_normal(R.shape)
    kind = 1 + np.arange(natoms, dtype=np.int32) % types
    out = []
    for lib in (gpu, oracle):
        md = lib.system(8, 1, rc, 0.4, natoms, kind, np.ones(types), None)
        for t in range(1, types + 1):
            lib.EmDee_set_pair_model(md, t, t, lib.EmDee_pair_lj_cut(1.0, 1.0), 0.0)
        lib.upload(md, "box", np.array([L]))
        lib.upload(md, "coordinates", R)
        lib.random_momenta(md, 1.0, True, 11)
        for _ in range(6):
            lib.boost(md, 1.0, 0.0, 0.0025)
            lib.displace(md, 1.0, 0.0, 0.005)
            lib.boost(md, 1.0, 0.0, 0.0025)
        out.append((lib.download(md, "forces", (natoms, 3)), md.Energy.Potential, md.Builds))
    (Fg, Ug, Bg), (Fo, Uo, Bo) = out
    assert Bg == Bo
    # 1e-14 of a box length of 54 in a separation of 0.8, times the 13 of a force's slope, grown twofold in 6 steps
    assert np.max(np.abs(Fg - Fo)) <= 1e-11 * np.max(np.abs(Fo))
    assert Ug == pytest.approx(Uo, rel=1e-11)
