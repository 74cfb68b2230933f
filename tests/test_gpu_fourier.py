"""The Bloch sum over pairs (R, -R) on the matrix cores against the plain sum
over R, at the edges of its tiles: 16 or 32 k-points, 64 elements, 4 pairs."""
import numpy as np
import pytest

import rustb_amd as ra
from oracle import oracle as O
from rustb_amd.model import synth_model

pytestmark = pytest.mark.gpu


def model(dim, n, n_R, seed, lone):
    """n_R stored vectors: 0, then R and -R in turn (the last pairless for an
    even n_R), or no two opposite with lone; the hoppings are not Hermitian."""
    g = np.random.default_rng(seed)
    grid = np.stack([x.reshape(-1) for x in np.meshgrid(*[np.arange(-4, 5)] * dim, indexing="ij")], axis=1)
    half = g.permutation(grid[len(grid) // 2 + 1:])
    if lone:
        rest = half[: n_R - 1] * g.choice([-1, 1], n_R - 1)[:, None]
    else:
        rest = np.stack([half, -half], axis=1).reshape(-1, dim)[: n_R - 1]
    hamR = np.vstack([np.zeros((1, dim), int), rest]).astype(np.int64)
    ham = g.standard_normal((len(hamR), n, 2 * n)).view(np.complex128)
    lat = np.eye(dim) * 2.0 + g.uniform(-0.3, 0.3, (dim, dim))
    orb = g.random((n, dim))
    return ra.Model.from_arrays(lat, orb, False, hamR, ham), lat, orb, hamR, ham


@pytest.mark.parametrize("dim,n,n_R,nk,lone", [
    (1, 1, 1, 1, False), (1, 2, 3, 15, False), (2, 3, 8, 16, False), (2, 7, 9, 17, True), (3, 8, 10, 33, False),
    (3, 9, 64, 31, False), (2, 17, 25, 65, False), (3, 33, 67, 2, False), (3, 24, 30, 1900, True),
    (3, 40, 12, 700, False)])
def test_paired_sum_at_tile_edges(dim, n, n_R, nk, lone):
    m, lat, orb, hamR, ham = model(dim, n, n_R, 100 * n + nk, lone)
    g = np.random.default_rng(nk)
    k, dirs = g.uniform(-1.0, 1.0, (nk, dim)), g.standard_normal((3, dim))
    some = np.unique(np.r_[0, nk - 1, g.integers(0, nk, 20)])
    U = np.exp(2j * np.pi * (k[some] @ hamR.T))
    H = np.einsum("kr,rij->kij", U, ham)
    scale = np.abs(ham).sum(0).max()
    # a term's phase and product (|2 pi k.R| <= 76), then n_R additions
    tol = np.finfo(float).eps * (n_R + 160) * scale
    for gauge in ("lattice", "atom"):
        P = np.ones((len(some), n, n))
        if gauge == "atom":
            f = np.exp(2j * np.pi * (k[some] @ orb.T))
            P = f.conj()[:, :, None] * f[:, None, :]
        assert np.abs(m.gen_ham_all(k, gauge)[some] - H * P).max() <= tol
        for n_p in (1, 2, 3):
            V, Hv = m.gen_v_projected_all(k, gauge, dirs[:n_p])
            assert np.abs(Hv[some] - H * P).max() <= tol
            for p in range(n_p):
                w, t = hamR @ lat @ dirs[p], orb @ lat @ dirs[p]
                X = 1j * np.einsum("kr,rij->kij", U * w, ham)
                if gauge == "atom":
                    X = X + 1j * (t[None, :] - t[:, None]) * H
                assert np.abs(V[some, p] - X * P).max() <= tol * (np.abs(w).max() + 2 * np.abs(t).max() + 1)


@pytest.mark.parametrize("mesh,n", [((1, 1), 2), ((3, 2), 3), ((4, 1, 2), 8), ((5, 2, 3), 9), ((16, 2), 11), ((17, 3), 4)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("mixed", 1e-6)])
def test_mesh_sum_at_tile_edges(mesh, n, precision, tol):
    """The uniform mesh's last pass (4 k-points per thread, 64 elements), with
    the velocities one by one (fp64) and as one operator (mixed)."""
    m = synth_model(2, len(mesh), False, n, 1, 40 + n)
    o = O.model_from_arrays(m.lat, m.orb, m.spin, m.hamR, m.ham)
    dirs = np.eye(len(mesh))[:2] + 0.1
    p = ra.Parameters(kmesh=mesh, direction=dirs, mu=np.array([-0.2, 0.3]), eta=0.05, T=np.array([900.0]),
                      precision=precision)
    got = m.hall_conductivity(p).conductivity
    ref = O.hall_conductivity_direct(o, list(mesh), dirs, np.array([-0.2, 0.3]), 900.0, 0.05)
    # as the products' tests: an eigenvector's error over the gap, times |v|^2 / eta^2
    assert np.abs(got - ref).max() <= tol * max(np.abs(ref).max(), 1e-2)
