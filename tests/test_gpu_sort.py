"""The cell sort and permutation of a list build against the oracle, around
the sizes up to which one workgroup sorts (16,384 atoms, 16,384 cells: 25 to a
side), with atoms in scrambled order and in several images of the box."""
import numpy as np
import pytest

import bench

pytestmark = pytest.mark.gpu

RC, SKIN = 2.5, 0.3


# cells to a side: floor(3 L / (rc + skin)), at least 7
@pytest.mark.parametrize("natoms,side", [(2, 6.0), (900, 9.9), (1025, 0.0), (2000, 23.8), (2000, 24.4), (16384, 0.0),
                                         (16385, 0.0)])
def test_builds_in_scrambled_order(gpu, oracle, natoms, side):
    R, L = bench.fcc_lattice(natoms, natoms / side**3 if side else 0.8442)
    rng = np.random.default_rng(17)
    R = R[rng.permutation(natoms)] + 0.04 * rng.standard_normal((natoms, 3)) + L * rng.integers(-2, 3, (natoms, 3))
    out = []
    for lib in (gpu, oracle):
        md = lib.system(1, 1, RC, SKIN, natoms, None, None, None)
        lib.EmDee_set_pair_model(md, 1, 1, lib.EmDee_pair_lj_cut(1.0, 1.0), 0.0)
        lib.upload(md, "box", np.array([L]))
        lib.upload(md, "coordinates", R)
        F0 = lib.download(md, "forces", (natoms, 3))
        lib.random_momenta(md, 1.2, True, 11)
        for _ in range(12):
            lib.boost(md, 1.0, 0.0, 0.004)
            lib.displace(md, 1.0, 0.0, 0.008)
            lib.boost(md, 1.0, 0.0, 0.004)
        out.append((F0, lib.download(md, "coordinates", (natoms, 3)), md.Energy.Potential, md.Builds))
    (Fg, Rg, Ug, Bg), (Fo, Ro, Uo, Bo) = out
    assert Bg == Bo and Bg >= (2 if natoms > 2 else 1)
    # up to 100 terms in another order, coordinates of several box lengths (1e-16 of 60 in a separation of 1, times
    # the 13 of a force's slope); 12 steps of 0.008 grow it a few times
    assert np.max(np.abs(Fg - Fo)) <= 2e-12 * max(1.0, np.max(np.abs(Fo)))
    assert np.max(np.abs(Rg - Ro)) <= 1e-10
    assert Ug == pytest.approx(Uo, rel=1e-10)
