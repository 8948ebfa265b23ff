"""Exact free rotation on the GPU against an independent integration: the
attitude matrix of every body advanced with its space-frame angular momentum
fixed (Runge-Kutta of order 4, many steps).  The angle max|omega| dt runs from
the power series' smallest steps over one and several substeps (0.16 each, at
most eight) to the closed form beyond them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def inertia_tensors(R, m):
    d = R - ((m[:, None] * R).sum(1) / m.sum())[:, None]
    return d, (m[:, None, None] * ((d ** 2).sum(-1)[..., None, None] * np.eye(3) - d[..., :, None] * d[..., None, :])).sum(1)


def bodies(nb, nsites, seed):
    """nb bodies of nsites random sites each (three sites: flat bodies), on a lattice of centres, and atom momenta."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(nb ** (1.0 / 3.0)))
    g = np.stack(np.meshgrid(*(np.arange(m),) * 3, indexing="ij"), -1).reshape(-1, 3)[:nb]
    mass = np.array([1.0, 4.0])
    types = np.tile(1 + np.arange(nsites, dtype=np.int32) % 2, nb)
    # moments apart from one another: the set-up's analytic eigensolver loses digits with their relative gap
    shape = rng.uniform(-1.0, 1.0, size=(40 * nb, nsites, 3))
    w = np.linalg.eigvalsh(inertia_tensors(shape, mass[types[:nsites] - 1])[1])
    shape = shape[np.minimum(np.min(np.diff(w, axis=1), axis=1), w[:, 0]) > 0.15 * w[:, 2]][:nb]
    R = (4.0 * (g + 0.5))[:, None, :] + shape
    P = rng.standard_normal((nb, nsites, 3))
    return R, P, mass, types, 4.0 * m


def free_rotation(R, P, m, angle, n=3000):
    """Member positions after a time dt with the largest |omega| dt of any principal component equal to `angle`."""
    d, inertia = inertia_tensors(R, m)
    M, c = m.sum(), R[:, 0] - d[:, 0]
    inv, L, p = np.linalg.inv(inertia), np.cross(d, P).sum(1), P.sum(1)
    w, v = np.linalg.eigh(inertia)
    dt = angle / np.max(np.abs(np.einsum("bji,bj->bi", v, L) / w))

    def rate(A):
        om = np.einsum("bij,bjk,blk,bl->bi", A, inv, A, L)
        return np.cross(om[:, None, :], A.transpose(0, 2, 1)).transpose(0, 2, 1)

    A, h = np.broadcast_to(np.eye(3), inertia.shape).copy(), dt / n
    for _ in range(n):
        k1 = rate(A)
        k2 = rate(A + 0.5 * h * k1)
        k3 = rate(A + 0.5 * h * k2)
        A = A + h / 6.0 * (k1 + 2.0 * k2 + 2.0 * k3 + rate(A + h * k3))
    return (c + dt / M * p)[:, None] + np.einsum("bij,bkj->bki", A, d), dt


@pytest.mark.parametrize("nsites", [3, 4])
@pytest.mark.parametrize("angle", [1e-5, 0.05, 0.16, 0.161, 0.7, 1.27, 1.3, 2.5])
def test_free_rotation(gpu, nsites, angle):
    nb = 130                                  # 260 lanes: a block and a remainder
    R, P, mass, types, L = bodies(nb, nsites, 7)
    ref, dt = free_rotation(R, P, mass[types[:nsites] - 1], angle)
    md = gpu.system(1, 1, 0.4 * L, 0.05 * L, nb * nsites, types, mass, np.repeat(np.arange(1, nb + 1, dtype=np.int32), nsites))
    for t in (1, 2):
        gpu.EmDee_set_pair_model(md, t, t, gpu.EmDee_pair_none(), 0.0)
    gpu.upload(md, "box", np.array([L]))
    gpu.upload(md, "coordinates", R.reshape(-1, 3))
    gpu.upload(md, "momenta", P.reshape(-1, 3))
    k0 = md.Kinetic.Total
    gpu.displace(md, 1.0, 0.0, dt)
    out = gpu.download(md, "coordinates", (nb * nsites, 3)).reshape(nb, nsites, 3)
    # the reference's own error is below 1e-13 (steps of 1e-3 rad: (1e-3)^4 2.5 / 120, and 3,000 roundings of 1e-16);
    # the body frame of the set-up's analytic eigensolver is good to 1e-10, at a distance of 2 from the centre
    assert np.max(np.abs(out - ref)) < 2e-10
    # a zero kick reads the kinetic energy, which the rotation conserves whatever the error of the frame: a few
    # roundings per substep (the closed form adds its quotients by moment differences, 1e-16 / 0.15)
    gpu.boost(md, 0.0, 0.0, 1.0)
    assert md.Kinetic.Total == pytest.approx(k0, rel=1e-13)
    P1 = gpu.download(md, "momenta", (nb * nsites, 3)).reshape(nb, nsites, 3)
    m = mass[types[:nsites] - 1]
    about = lambda r, p: np.cross(r - ((m[:, None] * r).sum(1) / m.sum())[:, None], p).sum(1)  # noqa: E731
    assert np.max(np.abs(about(out, P1) - about(R, P))) < 2e-10 * np.max(np.abs(P)) * 16.0
