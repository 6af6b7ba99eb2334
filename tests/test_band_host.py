"""The routines of the 1D eigenpair kernel and of the orbital response (qex_amd/csrc/band.h, band_wave.h, eigen1d.h)
on emulated lanes, against LAPACK on random 1D Kohn-Sham Hamiltonians (CPU only)."""

import ctypes

import numpy as np
import pytest

from oracle import od as O


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


class Band:
    """T + diag(v) on a grid, and the device routines on it."""

    def __init__(self, lib, grids, v):
        dx = O.get_dx(grids)
        s = -0.5 / (dx * dx)
        self.lib, self.N = lib, len(v)
        self.b, self.c = ctypes.c_double(s * (4.0 / 3.0)), ctypes.c_double(s * (-1.0 / 12.0))
        self.a = np.ascontiguousarray(s * -2.5 + v)
        self.H = O.get_kinetic_matrix(grids) + np.diag(v)
        self.hnorm = np.abs(self.a).max() + 2 * (abs(self.b.value) + abs(self.c.value))

    def count(self, x):
        return self.lib.host_sturm(self.N, _p(self.a), self.b, self.c, ctypes.c_double(x))

    def wave_count(self, x):
        return self.lib.host_wave_count(self.N, _p(self.a), self.b, self.c, ctypes.c_double(x))

    def solve(self, y, x, how="host_wave_solve"):
        y = np.array(y, dtype=np.float64)
        getattr(self.lib, how)(self.N, _p(self.a), _p(y), self.b, self.c, ctypes.c_double(x))
        return y

    def refine(self, y, j, lo, hi, check):
        y, rho = np.array(y, dtype=np.float64), np.zeros(1)
        ok = self.lib.host_refine(self.N, _p(self.a), _p(y), self.b, self.c, j, ctypes.c_double(lo), ctypes.c_double(hi),
                                  int(check), _p(rho))
        return bool(ok), rho[0], y

    def bracket(self, j):
        """The device's bracket width by bisection on the two-sided counts."""
        off = 2 * (abs(self.b.value) + abs(self.c.value))
        lo, hi = self.a.min() - off, self.a.max() + off
        while hi - lo > 1e-9 * max(1.0, abs(0.5 * (lo + hi))) + 64 * 2.2e-16 * self.hnorm:
            mid = 0.5 * (lo + hi)
            lo, hi = (lo, mid) if self.count(mid) > j else (mid, hi)
        return lo, hi


def _hamiltonians(lib, trials):
    rng = np.random.default_rng(0)
    for trial in range(trials):
        grids = O.h2_config_grid() if trial % 2 else np.linspace(-10, 10, 201 + trial % 3)
        A = int(rng.integers(1, 5))
        loc, Z = np.sort(rng.uniform(-4, 4, A)), rng.integers(1, 5, A)
        if trial % 6 == 0:
            loc, Z = np.array([-4.0, 4.0]), np.array([2, 2])  # nearly degenerate pairs
        v = O.get_atomic_chain_potential(grids, loc, Z, O.exponential_coulomb)
        if trial % 4 == 1:
            v = v + rng.normal(0, 0.2, len(v))
        yield trial, Band(lib, grids, v)


def _start(N, j):
    return np.sin(1.3 * np.arange(N) + 0.7 * j + 0.1)


def test_lowest_eigenpairs_match_lapack(lanes_lib):
    """Two-sided counts to a bracket of 1e-9, then the two twisted solves at its middle: eigenvalues to 1e-11,
    vectors to 1e-8 where the neighbours are 1e-6 away."""
    for trial, m in _hamiltonians(lanes_lib, 12):
        w, V = np.linalg.eigh(m.H)
        for j in range(5):
            lo, hi = m.bracket(j)
            x = m.solve(_start(m.N, j), 0.5 * (lo + hi), "host_twisted")
            assert abs(x @ m.H @ x - w[j]) < 1e-11
            if min(abs(w[j] - w[i]) for i in range(6) if i != j) > 1e-6:
                assert min(np.linalg.norm(x - V[:, j]), np.linalg.norm(x + V[:, j])) < 1e-8, (trial, j)


def test_counts_match_the_spectrum(lanes_lib):
    """Shifts across the spectrum, none within rounding of an eigenvalue: the two-sided count, and one wave's
    substructured factorisation."""
    for trial, m in _hamiltonians(lanes_lib, 6):
        w = np.linalg.eigvalsh(m.H)
        for x in np.concatenate([np.linspace(w[0] - 1, w[-1] + 1, 60), w[:5] - 1e-9, w[:5] + 1e-9]):
            if np.abs(w - x).min() > 64 * 2.2e-16 * m.hnorm:
                assert m.count(x) == m.wave_count(x) == int((w < x).sum())


@pytest.mark.parametrize("N", [5, 6, 7, 63, 64, 65, 127, 191, 192, 193, 257, 513, 1024])
def test_solves_match_dense(lanes_lib, N):
    """(A - sigma)^-1 y by one wave (rows a lane: odd, at least 5; sizes where a lane has no rows, part of its
    rows and all of them) and by the pivoted elimination, at shifts between eigenvalues: backward error
    |(A - sigma) x - y| <= 1e-11 |A| |x| (the growth of the unpivoted elimination included), the pivoted one's
    100 eps."""
    rng = np.random.default_rng(N)
    grids = 0.1 * (np.arange(N) - N // 2)
    m = Band(lanes_lib, grids, -2.0 * np.exp(-grids**2) + 0.1 * rng.standard_normal(N))
    w = np.linalg.eigvalsh(m.H)
    for j in (0, min(2, N - 2)):
        x = 0.5 * (w[j] + w[j + 1])
        y = rng.standard_normal(N)
        for how, tol in (("host_wave_solve", 1e-11), ("host_pivoted_solve", 100 * 2.2e-16)):
            z = m.solve(y, x, how)
            assert np.linalg.norm(m.H @ z - x * z - y) <= tol * m.hnorm * np.linalg.norm(z) + 1e-13 * np.linalg.norm(y)


@pytest.mark.parametrize("N", [5, 6, 65, 257, 513])
def test_solves_at_an_eigenvalue(lanes_lib, N):
    """The shift at an eigenvalue (the orbital response): the solution outside the eigenvector's direction, after
    one projection, against the pseudo-inverse; pivoted as the fallback takes it, one wave as it starts."""
    rng = np.random.default_rng(N)
    grids = 0.1 * (np.arange(N) - N // 2)
    m = Band(lanes_lib, grids, -2.0 * np.exp(-grids**2))
    w, V = np.linalg.eigh(m.H)
    p = V[:, 0]
    y = rng.standard_normal(N)
    y -= p * (p @ y)
    ref = V[:, 1:] @ ((V[:, 1:].T @ y) / (w[1:] - w[0]))
    for how in ("host_wave_solve", "host_pivoted_solve"):
        z = m.solve(y, p @ m.H @ p, how)
        z -= p * (p @ z)
        # rounding of the operator over the gap
        assert np.linalg.norm(z - ref) <= 1e3 * 2.2e-16 * m.hnorm / (w[1] - w[0]) * np.linalg.norm(ref)


def test_refined_eigenvalues_match_lapack(lanes_lib):
    """One wave's Rayleigh-quotient steps: inside a bracket of one eigenvalue, and from a vector close to the
    wanted one (as the last iteration's orbital)."""
    rng = np.random.default_rng(5)
    for trial, m in _hamiltonians(lanes_lib, 8):
        w, V = np.linalg.eigh(m.H)
        for j in range(4):
            near = min(abs(w[j] - w[i]) for i in range(6) if i != j)
            if near > 0.1:
                ok, rho, _ = m.refine(_start(m.N, j), j, w[j] - 0.01, w[j] + 0.008, False)
                assert ok and abs(rho - w[j]) < 1e-11
                y = V[:, j] + 1e-4 * rng.standard_normal(m.N) / np.sqrt(m.N)
                ok, rho, _ = m.refine(y / np.linalg.norm(y), j, w[0] - 1, w[-1] + 1, True)
                assert ok and abs(rho - w[j]) < 1e-11
                # the same vector asked for as another pair
                assert not m.refine(y / np.linalg.norm(y), j + 1, w[0] - 1, w[-1] + 1, True)[0]


@pytest.mark.parametrize("distance", [7.2, 7.8, 8.4, 9.0])
def test_mixtures_of_a_close_pair_are_not_refined(lanes_lib, distance):
    """Two wells whose lowest pair is split by 3e-10 .. 1e-7, and a vector between the two states (an orbital
    of an earlier iteration): its residual is half the splitting and its quotient lies between the levels, so it
    must not pass for either of them.  What passes is within 1e-11 of the value and 64 roundings of the operator."""
    grids = 0.1 * (np.arange(401) - 200)
    v = -6.0 * (np.exp(-((grids - distance / 2) ** 2)) + np.exp(-((grids + distance / 2) ** 2)))
    m = Band(lanes_lib, grids, v)
    w, V = np.linalg.eigh(m.H)
    split = w[1] - w[0]
    assert 3e-10 < split < 1e-7
    tol = 1e-11 * abs(w[0]) + 64 * 2.2e-16 * m.hnorm + 1e-12  # (1e-12: LAPACK's own)
    for angle in (0.25, 0.15, 0.4):
        y = np.cos(angle * np.pi) * V[:, 0] + np.sin(angle * np.pi) * V[:, 1]
        for j in (0, 1):
            ok, rho, _ = m.refine(y, j, w[0] - 1, w[-1] + 1, True)
            assert not ok or abs(rho - w[j]) < tol
    for j in (0, 1):
        ok, rho, _ = m.refine(V[:, j], j, w[0] - 1, w[-1] + 1, True)
        assert not ok or abs(rho - w[j]) < tol
