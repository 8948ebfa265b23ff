"""Neighbour lists of the batched HMC kernel at the edges of their packets of
eight entries and past their capacity, against the reference-API replay on
the oracle."""
import numpy as np
import pytest

import hmc_ref
from emdee_amd.hmc import BatchedHMC

pytestmark = pytest.mark.gpu

DT, SEED, CYCLES = 0.004, 41, 2


def cluster(n, box, seed):
    """n atoms on a jittered cubic lattice of spacing 1.12 in a corner of the
    box, across its faces."""
    m = int(np.ceil(n ** (1.0 / 3.0) - 1e-9))
    g = np.stack(np.meshgrid(*(np.arange(m),) * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    return 1.12 * (g - 0.4 * m) + np.random.default_rng(seed).uniform(-0.02, 0.02, size=(n, 3))


# (atoms of each replica, box side): all atoms of the small clusters are each
# other's neighbours (one less or more than a packet, whole packets); the
# clusters of 100 and 130 atoms hold up to twice the 32 entries
# that the density of their box gives a list
CASES = [([2, 8, 9, 10, 16, 17, 18, 25], 9.0), ([100, 3, 130], 16.0)]


@pytest.mark.parametrize("nsteps", [1, 2, 7])
@pytest.mark.parametrize("sizes,box", CASES)
def test_lists_at_packet_edges(gpu, oracle, sizes, box, nsteps):
    # The plain form evaluates the reference's pair terms in FP64 (1e-13 of a
    # force of about 1e2 in another order), which 14 steps of 0.004 carry to
    # 1e-12 in coordinates and, by the forces, 1e-10 in energies; the mixed
    # form's FP32 pair terms are off by 1e-6 of the largest ones.
    N = np.array(sizes, dtype=np.int32)
    L, T = np.full(len(N), box), np.full(len(N), 0.3)
    Rs = [cluster(int(n), box, 5 + k) for k, n in enumerate(N)]
    Ro, Uo, Ao, _ = hmc_ref.replay(oracle, oracle, N, L, T, Rs, CYCLES, dt=DT, nsteps=nsteps, seed=SEED)
    for precision in (0, 1):
        h = BatchedHMC(gpu, N, L, T, Rs, dt=DT, nsteps=nsteps, seed=SEED, precision=precision)
        h.run(launches=2, cycles=1)
        R, U, A, _ = h.state()
        h.close()
        same = np.asarray(A) == np.asarray(Ao)
        assert np.all(same) if precision == 0 else np.sum(~same) <= 1
        tolR, tolU = (1e-9, 1e-8) if precision == 0 else (1e-4, 1e-3)
        for k in np.nonzero(same)[0]:
            assert np.max(np.abs(R[k] - Ro[k])) < tolR, (sizes[k], precision)
            assert abs(U[k] - Uo[k]) < tolU * max(1.0, abs(Uo[k])), (sizes[k], precision)
