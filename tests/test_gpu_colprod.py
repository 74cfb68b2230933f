"""The on-chip products U^H X U at the edges of their 16-column tiles (every
tile count from 1 to 8, sizes just below, at and above a tile), against the
oracle: the term-by-term band sum (fp64, metric, spin current) and the
one-product band sum (mixed)."""
import numpy as np
import pytest

import rustb_amd as ra
from oracle import oracle as O
from rustb_amd.model import synth_model

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 32, 33, 47, 49, 64, 65, 81, 96, 97, 112, 113, 127, 128]


def pair(n, spin=False):
    m = synth_model(1, 3, spin, n // 2 if spin else n, 1, 300 + n, scale=0.5, decay=1.0)
    return m, O.model_from_arrays(m.lat, m.orb, m.spin, m.hamR, m.ham)


@pytest.mark.parametrize("n", EDGES)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_omega_at_tile_edges(n, precision):
    m, o = pair(n)
    ks = np.random.default_rng(n).random((5, 3))
    d = np.array([[1.0, 0.2, 0.0], [0.0, 1.0, -0.3]])
    p = ra.Parameters(kmesh=(1, 1, 1), direction=d, mu=np.array([0.0]), eta=0.05, precision=precision)
    om, E = m.berry_curvature_on(ks, p)
    ob, Eb = O.berry_curvature_batch(o, ks, d, 0.05)
    # Omega's error is an eigenvector's (rounding over the gap; fp64 ~1e-15,
    # mixed ~1e-11 of the spectrum) times |v|^2 / eta^2: a few 1e2 of Omega's scale
    tol = 1e-10 if precision == "fp64" else 1e-7
    assert np.abs(E - Eb).max() < (1e-11 if precision == "fp64" else 1e-9)
    assert np.abs(om - ob).max() <= tol * max(np.abs(ob).max(), 1e-3)


@pytest.mark.parametrize("n", [2, 16, 34, 66, 98, 128])
def test_spin_current_and_metric_at_tile_edges(n):
    m, o = pair(n, spin=True)
    ks = np.random.default_rng(n).random((4, 3))
    d = np.eye(3)[:2]
    p = ra.Parameters(kmesh=(1, 1, 1), direction=d, mu=np.array([0.0]), eta=0.05, spin="Y")
    om, E = m.berry_curvature_on(ks, p)
    ob, Eb = O.berry_curvature_batch(o, ks, d, 0.05, "Y")
    assert np.abs(om - ob).max() <= 1e-10 * max(np.abs(ob).max(), 1e-3)
    p.spin = None
    r = m.quantum_geometry_on(ks, p)
    for i, k in enumerate(ks):
        g = O.quantum_geometry_at(o, k, d, 0.05)
        assert np.abs(r.metric[i] - g[0]).max() <= 1e-10 * max(np.abs(g[0]).max(), 1e-3)


@pytest.mark.parametrize("mesh,n_mu,T", [((1, 1), 1, 0.0), ((7, 9), 8, 300.0), ((8, 8), 9, 0.0), ((13, 5), 17, 900.0),
                                         ((50, 41), 3, 300.0)])
def test_hall_sums_at_block_edges(mesh, n_mu, T):
    """The occupation sums in blocks of 64 k-points and 8 chemical potentials,
    and the row sums above and below 32 blocks."""
    m = synth_model(3, 2, False, 3, 1, 17, n_R_target=9)
    o = O.model_from_arrays(m.lat, m.orb, m.spin, m.hamR, m.ham)
    mu = np.linspace(-1.0, 1.3, n_mu)
    p = ra.Parameters(kmesh=mesh, direction=np.eye(2), mu=mu, eta=0.05, T=np.array([T]))
    got = m.hall_conductivity(p).conductivity
    ref = O.hall_conductivity_direct(o, list(mesh), np.eye(2), mu, T, 0.05)
    assert np.abs(got - ref).max() <= 1e-10 * max(np.abs(ref).max(), 1e-3)


@pytest.mark.parametrize("mesh,n_mu", [((90, 91), 9), ((300, 220), 41), ((171, 181), 70)])
def test_hall_sums_over_chunks(mesh, n_mu, monkeypatch):
    """The occupation sums in blocks of 64 and of 256 k-points, in one chunk
    and added up over several, for the curvature, the metric and the dipole."""
    m = synth_model(3, 2, False, 3, 1, 17, n_R_target=9)
    p = ra.Parameters(kmesh=mesh, direction=np.eye(2), mu=np.linspace(-1.0, 1.3, n_mu), eta=0.05, T=np.array([300.0]))
    d = ra.Parameters(kmesh=mesh, direction=np.array([[1.0, 0.0], [0.0, 1.0], [1.0, 1.0]]), mu=p.mu, eta=0.05, T=p.T)

    def call():
        g = m.quantum_geometry(p)
        return [m.hall_conductivity(p).conductivity, g.metric, g.berry_curvature, m.extrinsic_nonlinear_hall(d).conductivity]

    one = call()
    monkeypatch.setenv("RTB_WORKSPACE_MB", "6")
    for a, b in zip(one, call()):
        # sums of nk terms in another order
        assert np.abs(a - b).max() <= 1e-11 * max(np.abs(a).max(), 1e-3)


@pytest.mark.parametrize("mesh,En", [((1, 1), 1), ((5, 7), 256), ((33, 31), 257), ((200, 90), 801)])
def test_dos_at_block_edges(mesh, En):
    """The DOS in blocks of 64 to 2048 eigenvalues and 256 energies."""
    m = ra.workloads.graphene()
    o = O.model_from_arrays(m.lat, m.orb, m.spin, m.hamR, m.ham)
    E, rho = m.dos(mesh, -4.0, 4.0, En, 0.05)
    Er, rr = O.dos(o, list(mesh), -4.0, 4.0, En, 0.05)
    # sums of nk positive terms in another order: nk eps of the result
    assert np.abs(rho - rr).max() <= 1e-11 * max(np.abs(rr).max(), 1e-300)


def test_dos_with_more_energies_than_workgroups_of_a_launch():
    """2^24 + 1 energies over 32 blocks of eigenvalues: a workgroup per energy
    would be 2^32 threads, more than a launch holds."""
    m = ra.workloads.graphene()
    E, rho = m.dos((128, 256), -4.0, 4.0, 2**24 + 1, 0.05)
    Er, rr = m.dos((128, 256), -4.0, 4.0, 2**8 + 1, 0.05)
    np.testing.assert_allclose(E[:: 2**16], Er, rtol=0, atol=1e-14)
    # the same terms in another order: nk eps, and the energies' rounding over sigma
    np.testing.assert_allclose(rho[:: 2**16], rr, rtol=0, atol=1e-11 * rr.max())


def test_more_k_points_than_a_launch_holds(monkeypatch):
    """8200 x 8200 k-points of one band fit the workspace at once, but at a
    workgroup of 64 threads each they are more than 2^32 threads."""
    m = synth_model(3, 2, False, 1, 1, 5, n_R_target=9)
    one = m.dos((8200, 8200), -2.0, 2.0, 11, 0.3)[1]
    monkeypatch.setenv("RTB_WORKSPACE_MB", "2000")
    many = m.dos((8200, 8200), -2.0, 2.0, 11, 0.3)[1]
    # sums of nk positive terms in another order
    np.testing.assert_allclose(one, many, rtol=1e-11)
