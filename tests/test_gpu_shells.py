"""Lists ordered by distance shells (16-lane build) against the oracle while
the displacement grows through every shell, in both forms, with filters, an
inner cutoff and a box that changes; and a cluster whose shells overflow."""
import ctypes

import numpy as np
import pytest

import bench
from emdee_amd.water_box import KB, KCOUL, water_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixed", [0, 1])
def test_displaced_by_parts_of_the_skin(gpu, oracle, mixed):
    """Atoms moved by up to 0, 1/10, ... of half the skin from the build positions: no rebuild until the last."""
    nmol, skin = 700, 2.0
    N = 3 * nmol
    (mg, cfg), (mo, _) = (water_system(lib, nmol, 3, rc=8.0, skin=skin, coul="damped", alpha=0.3) for lib in (gpu, oracle))
    gpu.EmDeeGPU_set_precision(mg, mixed)
    rng = np.random.default_rng(2)
    u = rng.standard_normal((nmol, 3))
    u = np.repeat(u / np.linalg.norm(u, axis=1, keepdims=True), 3, axis=0)
    for md in (mg, mo):
        md.Options.AutoBodyUpdate = False
    for f in (0.0, 0.1, 0.24, 0.26, 0.45, 0.55, 0.7, 0.8, 0.95, 1.3):
        F = []
        for lib, md in ((gpu, mg), (oracle, mo)):
            lib.upload(md, "coordinates", cfg["R"] + 0.5 * skin * f * u)
            F.append(lib.download(md, "forces", (N, 3)))
            lib.compute_forces(md)
        assert mg.Builds == mo.Builds
        err = np.max(np.abs(F[0] - F[1])) / np.max(np.abs(F[1]))
        assert err < (1e-5 if mixed else 1e-12), f
        if not mixed:   # (the mixed form bounds the force error; this energy is a small difference of large sums)
            assert mg.Energy.Potential == pytest.approx(mo.Energy.Potential, rel=1e-11)


def test_dynamics_with_box_scaling(gpu, oracle):
    """alpha != 0 scales coordinates and box together, so that an image moves with the box."""
    out = []
    for lib in (gpu, oracle):
        md, cfg = water_system(lib, 700, 3, rc=8.0, skin=2.0, coul="damped", alpha=0.3)
        lib.random_momenta(md, KB * 298.0, True, 5)
        rec = []
        for k in range(12):
            lib.boost(md, 1.0, 0.0, 0.5)
            lib.displace(md, 1.0, 1e-3 if k % 3 == 1 else 0.0, 1.0)
            lib.boost(md, 1.0, 0.0, 0.5)
            rec.append([md.Energy.Potential, md.Kinetic.Total, md.Builds])
        out.append(np.array(rec))
    np.testing.assert_allclose(out[0], out[1], rtol=1e-8)


@pytest.mark.parametrize("exclude", [False, True])
def test_shell_overflow(gpu, oracle, exclude):
    """A Gauss cluster at the box centre: atoms with far more shell entries than the build keeps apart."""
    rng = np.random.default_rng(4)
    R = np.concatenate([12.0 + 2.2 * rng.standard_normal((1500, 3)), rng.uniform(0.0, 24.0, (1500, 3))])
    N, L = len(R), 24.0
    F, E = [], []
    for lib in (gpu, oracle):
        md = lib.system(1, 1, 3.0, 2.0, N, None, None, None)
        lib.EmDee_set_pair_model(md, 1, 1, lib.EmDee_pair_softcore_cut(1.0, 1.0, 0.5), 0.0)
        if exclude:
            for k in range(1, 400, 2):
                lib.EmDee_ignore_pair(md, k, k + 1)
        lib.upload(md, "box", np.array([L]))
        lib.upload(md, "coordinates", R)
        for step in range(3):
            lib.upload(md, "coordinates", R + 0.3 * step * np.sin(np.arange(3 * N)).reshape(N, 3) / np.sqrt(3.0))
            F.append(lib.download(md, "forces", (N, 3)))
            lib.compute_forces(md)
            E.append(md.Energy.Potential)
        if lib is gpu:
            pairs = lib.neighbor_pairs(md)
            assert len(pairs) == len({tuple(p) for p in pairs.tolist()})
    for k in range(3):
        assert np.max(np.abs(F[k] - F[k + 3])) <= 1e-11 * np.max(np.abs(F[k + 3]))
        assert E[k] == pytest.approx(E[k + 3], rel=1e-11)
