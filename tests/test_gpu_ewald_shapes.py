"""The reciprocal sum's matrix form on the GPU against the oracle where its
shapes can go wrong: a sphere of a few vectors, exactly one and more than one
block of sixteen columns, one to three charged types (with an uncharged one
among them), groups with a remainder, and more charge groups than chunks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def ions(lib, n, ntypes, L, rc, accuracy, seed=3):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*(np.arange(m),) * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    R = (g + rng.uniform(0.2, 0.8, size=(n, 3))) * (L / m)
    types = 1 + np.arange(n, dtype=np.int32) % ntypes
    q = rng.uniform(0.5, 1.5, size=n) * np.where(np.arange(n) % 2 == 0, 1.0, -1.0)
    if ntypes == 3:
        q[types == 2] = 0.0
    md = lib.system(1, 1, rc, 0.05 * rc, n, types, np.ones(ntypes), None)
    for t in range(1, ntypes + 1):
        lib.EmDee_set_pair_model(md, t, t, lib.EmDee_pair_none(), 0.7 + 0.1 * t)
    lib.EmDee_set_coul_model(md, lib.EmDee_coul_long())
    lib.EmDee_set_kspace_model(md, lib.EmDee_kspace_ewald(accuracy))
    lib.upload(md, "charges", q)
    lib.upload(md, "coordinates", R)
    lib.upload(md, "box", np.array([L]))
    return md


# n, types, box / cutoff, accuracy; the largest index of the sphere is 1, 2, 15, 16, 22 and 11
@pytest.mark.parametrize("n,ntypes,ratio,accuracy", [(60, 1, 2.6, 0.5), (257, 2, 2.6, 0.2), (513, 1, 4.1, 1e-6),
                                                     (700, 3, 4.3, 1e-6), (300, 2, 6.0, 1e-6), (33400, 1, 9.7, 1e-2)])
def test_reciprocal_sum(gpu, oracle, n, ntypes, ratio, accuracy):
    rc = 1.0
    mg, mo = (ions(lib, n, ntypes, ratio * rc, rc, accuracy) for lib in (gpu, oracle))
    Fg, Fo = gpu.download(mg, "forces", (n, 3)), oracle.download(mo, "forces", (n, 3))
    # FP64 sums over the charges and the vectors in another order, the phases by powers: a few hundred roundings
    assert np.max(np.abs(Fg - Fo)) <= 1e-11 * np.max(np.abs(Fo))
    assert mg.Energy.Coulomb == pytest.approx(mo.Energy.Coulomb, rel=1e-11)
    assert mg.Virial == pytest.approx(mo.Virial, rel=1e-10)
    # the atoms' shares add up to the energy
    assert np.sum(gpu.atom_energies(mg, n)) == pytest.approx(mo.Energy.Potential, rel=1e-10)
