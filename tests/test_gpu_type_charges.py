"""Charged systems whose atoms of a type share one charge (read from LDS up to
eight types), have charges of their own, or have more types than LDS holds, in
the kernels of one and of several lanes per atom, against the oracle."""
import numpy as np
import pytest

from parity_util import build, fcc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms,types", [(864, 1), (864, 2), (864, 8), (864, 9), (70304, 3)])
@pytest.mark.parametrize("own", [False, True])
def test_charges(gpu, oracle, natoms, types, own):
    R, L = fcc(natoms, 0.7, jitter=0.05, seed=3)
    rng = np.random.default_rng(9)
    kind = (1 + rng.permutation(natoms) % types).astype(np.int32)
    of_type = np.where(np.arange(types) % 3 == 1, 0.0, rng.uniform(-1.0, 1.0, types))   # some types uncharged
    q = of_type[kind - 1]
    if own:
        q[natoms // 2] += 0.25          # one atom of its type differs
    models = [lambda lib, t=t: lib.EmDee_pair_lj_cut(1.0 + 0.05 * t, 1.0) if t % 4 != 2 else lib.EmDee_pair_none()
              for t in range(types)]
    out = []
    for lib in (gpu, oracle):
        md = build(lib, R, L, 2.5, 0.3, models, types=kind, masses=np.ones(types), charges=q,
                   coul=lambda lib: lib.EmDee_coul_damped(0.4), kcoul=1.0, threads=1 if lib is gpu else 8)
        out.append((lib.download(md, "forces", (natoms, 3)), md.Energy.Potential, md.Virial))
        if lib is gpu:
            lib.EmDeeGPU_set_precision(md, 1)
            lib.compute_forces(md)
            Fm = lib.download(md, "forces", (natoms, 3))
    (Fg, Ug, Wg), (Fo, Uo, Wo) = out
    # up to 80 terms in another order, coordinates of a box length of 46 at most (1e-16 of it in a separation of 0.8,
    # times the 13 of a force's slope); energies: random walk of 5e6 roundings on a sum a tenth of its terms
    assert np.max(np.abs(Fg - Fo)) <= 1e-12 * np.max(np.abs(Fo))
    assert Ug == pytest.approx(Uo, rel=1e-10)
    assert Wg == pytest.approx(Wo, rel=1e-10)
    assert np.linalg.norm(Fm - Fo) / np.linalg.norm(Fo) < 1e-5   # the mixed form's stated bound
