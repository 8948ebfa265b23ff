"""Launch shapes of the batched HMC in large dilute boxes: a shape fits when the cell table holds the grid that its
lists are built on (cells of side (rc + skin) / division, 6,144 cells), and every shape gives the same trajectories."""
import numpy as np
import pytest

import hmc_ref
from emdee_amd.hmc import BatchedHMC

pytestmark = pytest.mark.gpu

DT, SEED, CYCLES, NSTEPS = 0.004, 43, 2, 5


def scattered(n, box, seed):
    """n atoms in pairs 1.12 apart, the pairs on a lattice over the whole box."""
    m = int(np.ceil((n / 2) ** (1.0 / 3.0)))
    g = (np.stack(np.meshgrid(*(np.arange(m),) * 3, indexing="ij"), -1).reshape(-1, 3)[:n // 2] + 0.3) * (box / m)
    return np.concatenate([g, g + [1.12, 0.0, 0.0]]) + np.random.default_rng(seed).uniform(-0.02, 0.02, size=(n, 3))


# box side, shapes of cell division 1 and 2 that fit: cells per edge 17 at 25 (division 2; 20 of side rc / 2 would be
# too many) and at 50 (division 1), 18 at 25.9, 19 at 26.7
@pytest.mark.parametrize("box,fits", [(22.0, (1, 1)), (25.0, (1, 1)), (25.9, (1, 1)), (26.7, (1, 0)), (50.0, (1, 0))])
def test_large_boxes(gpu, oracle, box, fits):
    N = np.array([400, 300], dtype=np.int32)
    L, T = np.full(2, box), np.full(2, 0.3)
    Rs = [scattered(int(n), box, k) for k, n in enumerate(N)]
    h = BatchedHMC(gpu, N, L, T, Rs, dt=DT, nsteps=NSTEPS, seed=SEED, precision=0)
    t = h.tune()["timings_ms"]
    h.run(launches=CYCLES, cycles=1)
    R, U, A, _ = h.state()
    h.close()
    assert [int(x > 0) for x in t] == [fits[0]] * 3 + [fits[1]] * 3
    Ro, Uo, Ao, _ = hmc_ref.replay(oracle, oracle, N, L, T, Rs, CYCLES, dt=DT, nsteps=NSTEPS, seed=SEED)
    assert np.array_equal(A, Ao)
    # FP64 terms in another order, ten steps: as in the tests of the lists' packets
    assert np.max(np.abs(U - Uo)) < 1e-8 * max(1.0, np.max(np.abs(Uo)))
    assert all(np.max(np.abs(a - b)) < 1e-9 for a, b in zip(R, Ro))
