"""Vectors read back in chunks (65,536 to 262,144 doubles, through pinned
memory that the batched HMC reuses after 1,048,576) come back bit for bit."""
import numpy as np
import pytest

import bench
from emdee_amd.hmc import BatchedHMC, replica_set

pytestmark = pytest.mark.gpu


# one thread's, one block's, one chunk's and several chunks' edges (3 N doubles)
@pytest.mark.parametrize("natoms", [1, 341, 342, 10923, 21845, 21846, 87381, 87382, 262145, 400001])
def test_vectors(gpu, natoms):
    R, L = bench.fcc_lattice(natoms, 0.8442)
    rng = np.random.default_rng(natoms)
    R = R[rng.permutation(natoms)] + 0.04 * rng.standard_normal((natoms, 3)) + L * rng.integers(-1, 2, (natoms, 3))
    md = gpu.system(1, 1, 2.5, 0.3, natoms, None, None, None)
    gpu.EmDee_set_pair_model(md, 1, 1, gpu.EmDee_pair_lj_cut(1.0, 1.0), 0.0)
    gpu.upload(md, "box", np.array([max(L, 6.0)]))
    gpu.upload(md, "coordinates", R)
    P = rng.standard_normal((natoms, 3))
    gpu.upload(md, "momenta", P)
    gpu.compute_forces(md)                     # slots in cell order
    for _ in range(2):
        assert np.array_equal(gpu.download(md, "coordinates", (natoms, 3)), R)
        assert np.array_equal(gpu.download(md, "momenta", (natoms, 3)), P)
    gpu.upload(md, "forces", P)
    assert np.array_equal(gpu.download(md, "forces", (natoms, 3)), P)


@pytest.mark.parametrize("replicas,size", [(2, 108), (86, 4064), (130, 4100)])
def test_replicas(gpu, replicas, size):
    N, L, T, Rs = replica_set(replicas, seed=3, nmin=size, nmax=size)
    h = BatchedHMC(gpu, N, L, T, Rs, nsteps=1, precision=1)
    for _ in range(2):
        assert np.array_equal(np.concatenate(h.state()[0]), np.concatenate(Rs))
    h.close()
