"""Flat bands with a dispersive level close to them, in the diagonal form and
rotated to a dense matrix: spectra whose eigenvalue search cannot rely on
Newton steps (they crawl next to many equal levels)."""
import numpy as np
import pytest

import rustb_amd as ra

pytestmark = pytest.mark.gpu


def flat_model(n, rotated):
    """3n/4 levels at c, one at c + t(k) with t from 2e-5 to 0.1 of 2/n, the
    edges -1 and 1, the rest spread between; c lies 1e-4 of 2/n below a point
    -1 + 2 p/n (the eigenvalue search starts from those).  H(k) on a 1D chain."""
    g = np.random.default_rng(n)
    m, p, h = 3 * n // 4, n // 3, 2.0 / n
    c = -1.0 + p * h - 1e-4 * h
    lo, hi = 2e-5 * h, 0.1 * h
    d = np.concatenate([np.full(m, c), [c + 0.5 * (hi + lo), -1.0, 1.0], g.uniform(-1.0, 1.0, n - m - 3)])
    ham = np.zeros((3, n, n), np.complex128)
    ham[0] = np.diag(d)
    ham[1, m, m] = ham[2, m, m] = -0.25 * (hi - lo)  # c + t(k): t smallest at k = 0
    if rotated:
        q, _ = np.linalg.qr(g.standard_normal((n, 2 * n)).view(np.complex128))
        ham = q @ ham @ q.conj().T
        ham[0] = 0.5 * (ham[0] + ham[0].conj().T)
        ham[2] = ham[1].conj().T
    return ra.Model.from_arrays(np.eye(1), np.zeros((n, 1)), False, np.array([[0], [1], [-1]], np.int64), ham), ham


@pytest.mark.parametrize("rotated", [False, True])
@pytest.mark.parametrize("n", [32, 48, 64, 96, 128, 200])
def test_flat_bands(n, rotated):
    m, ham = flat_model(n, rotated)
    k = np.linspace(0.0, 0.5, 257) ** 2 * 2.0  # dense where the level is closest
    ph = np.exp(2j * np.pi * k)
    H = ham[0] + ph[:, None, None] * ham[1] + ph.conj()[:, None, None] * ham[2]
    ref = np.linalg.eigvalsh(H)
    # a backward stable solver's n eps ||H||, of both sides; the mixed form's
    # refined values to 1e-9.  A pair's residual is at least its eigenvalue's
    # error; the vectors of close levels, from inverse iteration, leave up to
    # 1e-11 (mixed 1e-9) themselves.
    tol = 4 * n * np.finfo(float).eps
    assert np.abs(m.solve_band_all(k[:, None], "fp64") - ref).max() <= tol
    assert np.abs(m.solve_band_all(k[:, None], "mixed") - ref).max() <= 1e-9
    for precision, t in (("fp64", tol), ("mixed", 1e-9)):
        E, V = m.solve_all(k[:, None], precision)
        assert np.abs(E - ref).max() <= t
        r = np.einsum("kij,knj->kni", H, V) - E[:, :, None] * V
        assert np.abs(r).max() <= 1e-8
