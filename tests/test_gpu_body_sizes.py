"""Rigid bodies of three to nine members (the kernels take members four at a
time, and two lanes place them) beside free atoms, against the oracle."""
import numpy as np
import pytest

from test_gpu_rotation import bodies

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 2])   # exact rotation by two lanes, no-squish by one
def test_sizes(gpu, oracle, mode):
    sizes = [3, 4, 5, 7, 8, 9]
    R, types, mol, P, n, L = [], [], [], [], 0, 24.0
    for layer, nsites in enumerate(sizes):
        r, p, mass, t, _ = bodies(36, nsites, 10 + layer)
        g = 4.0 * (np.stack(np.meshgrid(np.arange(6), np.arange(6), indexing="ij"), -1).reshape(-1, 2) + 0.5)
        centre = np.c_[g, np.full(36, 4.0 * layer + 2.0)]
        r = r - r.mean(1, keepdims=True) + centre[:, None, :]
        R.append(r.reshape(-1, 3)); P.append(p.reshape(-1, 3)); types.append(t)
        mol.append(np.repeat(n + np.arange(1, 37, dtype=np.int32), nsites))
        n += 36
    free = 4.0 * np.stack(np.meshgrid(*(np.arange(6),) * 3, indexing="ij"), -1).reshape(-1, 3)
    R.append(free.astype(float)); types.append(np.ones(216, dtype=np.int32)); mol.append(np.zeros(216, dtype=np.int32))
    P.append(np.random.default_rng(3).standard_normal((216, 3)))
    R, P = np.concatenate(R), np.concatenate(P)
    types, mol = np.concatenate(types).astype(np.int32), np.concatenate(mol).astype(np.int32)
    out = []
    for lib in (gpu, oracle):
        md = lib.system(1, 1, 4.0, 1.0, len(R), types, mass, mol)
        md.Options.RotationMode = mode
        for t in (1, 2):
            lib.EmDee_set_pair_model(md, t, t, lib.EmDee_pair_lj_cut(0.5, 0.8), 0.0)
        lib.upload(md, "box", np.array([L]))
        lib.upload(md, "coordinates", R)
        lib.upload(md, "momenta", P)
        rec = []
        for _ in range(8):
            lib.boost(md, 1.0, 0.0, 0.002)
            lib.displace(md, 1.0, 0.0, 0.004)
            lib.boost(md, 1.0, 0.0, 0.002)
            rec.append([md.Energy.Potential, md.Virial, md.Kinetic.Total, md.Kinetic.Rotational])
        out.append((np.array(rec), lib.download(md, "coordinates", (len(R), 3)), lib.download(md, "momenta", (len(R), 3))))
    (eg, Rg, Pg), (eo, Ro, Po) = out
    # principal axes good to 1e-10 of a body's size, turned by up to 0.1 rad and pulled by forces of slope 1e2
    np.testing.assert_allclose(eg, eo, rtol=1e-7)
    assert np.max(np.abs(Rg - Ro)) < 1e-8
    assert np.max(np.abs(Pg - Po)) < 1e-6
