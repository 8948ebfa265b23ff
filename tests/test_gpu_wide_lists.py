"""Long lists of systems past 131,072 atoms: the 16-lane streamed build, for
pairs that the distance alone decides and with excluded pairs, against the
oracle."""
import numpy as np
import pytest

import bench

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms,excluded", [(131073, 0), (140000, 1000), (530000, 10)])
def test_lists_of_large_systems(gpu, oracle, natoms, excluded):
    R, L = bench.fcc_lattice(natoms, 0.8442)
    rng = np.random.default_rng(23)
    R = R + 0.05 * rng.standard_normal((natoms, 3))
    out = []
    for lib in (gpu, oracle):
        md = lib.system(8, 1, 2.5, 0.3, natoms, None, None, None)
        lib.EmDee_set_pair_model(md, 1, 1, lib.EmDee_pair_lj_cut(1.0, 1.0), 0.0)
        for k in range(excluded):
            lib.EmDee_ignore_pair(md, 1 + k, 2 + k)
        lib.upload(md, "box", np.array([L]))
        lib.upload(md, "coordinates", R)
        out.append((lib.download(md, "forces", (natoms, 3)), md.Energy.Potential, md.Virial))
    (Fg, Ug, Wg), (Fo, Uo, Wo) = out
    # up to 100 terms in another order, coordinates of a box length L up to 86 (1e-16 of it in a separation of 0.8,
    # times the 13 of a force's slope)
    assert np.max(np.abs(Fg - Fo)) <= 5e-13 * np.max(np.abs(Fo))
    # random walk of 2e7 roundings: 5e-13
    assert Ug == pytest.approx(Uo, rel=1e-11)
    assert Wg == pytest.approx(Wo, rel=1e-10)
