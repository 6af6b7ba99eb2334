"""The device headers of the one-workgroup solvers on emulated lanes (tests/host/lanes: every thread of a
workgroup a fiber, exchanges and barriers as on the device, hardware reciprocals cut to their precision), against
LAPACK (CPU only)."""

import ctypes

import numpy as np
import pytest

EPS = np.finfo(float).eps


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _eigh(lanes_lib, A, nvec=1 << 30, solver="host_symeig"):
    A = np.ascontiguousarray(A, dtype=np.float64)
    n = len(A)
    w, Z, perm = np.zeros(n), np.zeros((n, n)), np.zeros(n, dtype=np.int32)
    getattr(lanes_lib, solver)(n, _p(A), nvec, _p(w), _p(Z), _p(perm))
    return w, Z, perm


def _check_eigh(lanes_lib, A, tol, unit=1.0):
    """Eigenvalues, residual and orthogonality within tol of the norm; A given in units of `unit`."""
    w, Z, _ = _eigh(lanes_lib, A * unit)
    ref = np.linalg.eigvalsh(A)
    norm = max(np.abs(ref).max(), 1e-300)
    w = w / unit
    assert np.abs(w - ref).max() <= tol * norm
    assert np.abs(A @ Z - Z * w).max() <= tol * norm
    assert np.abs(Z.T @ Z - np.eye(len(A))).max() <= tol


@pytest.mark.parametrize("n", [1, 2, 3, 8, 9, 16, 17, 33, 64, 65, 96])
def test_symeig_random(lanes_lib, n):
    """Sizes at the edges of the register patches and size classes.  The closest pair of such a matrix is
    1e-3 of the norm apart, where two inverse iterations leave eps / 1e-3 = 2e-13; 1e-12 with the sums over n."""
    A = np.random.default_rng(n).standard_normal((n, n))
    _check_eigh(lanes_lib, A + A.T, 1e-12)


@pytest.mark.parametrize("n", [3, 13, 15, 16, 22, 26, 33, 41])
@pytest.mark.parametrize("kind", ["ones", "pi", "bipartite"])
def test_symeig_rank_deficient_with_equal_entries(lanes_lib, n, kind):
    """Reduction leaves a block of rounding errors that keeps the symmetry of the matrix, so its columns shrink by
    1e-16 a reflector, through every magnitude where a square or its reciprocal is no normal number.
    Backward stability of n reflectors: 40 n eps."""
    if kind == "bipartite":
        A = np.zeros((n, n))
        A[: n // 2, n // 2:] = 1.0
        A += A.T
    else:
        A = np.full((n, n), 0.3 if kind == "ones" else np.pi)
    _check_eigh(lanes_lib, A, 40 * n * EPS)


@pytest.mark.parametrize("coupling", [1e-140, 1e-150, 1e-154, 1e-156, 1e-158, 1e-160, 1e-162, 1e-165, 1e-200])
def test_symeig_weakly_coupled_blocks(lanes_lib, coupling):
    """Two blocks joined by entries whose squares are near or below the smallest double (well separated
    fragments): the spectrum of the blocks."""
    rng = np.random.default_rng(4)
    A = np.zeros((12, 12))
    A[:6, :6], A[6:, 6:] = rng.standard_normal((6, 6)), rng.standard_normal((6, 6))
    A[6:, :6] = coupling * rng.standard_normal((6, 6))
    A = np.tril(A) + np.tril(A, -1).T
    _check_eigh(lanes_lib, A, 1e-13)
    # as the smallest example: two coupled pairs
    B = np.diag([1.0, 2.0, 3.0, 4.0])
    B[0, 1] = B[1, 0] = B[2, 3] = B[3, 2] = 0.3
    B[0, 2] = B[2, 0] = B[1, 3] = B[3, 1] = coupling
    _check_eigh(lanes_lib, B, 40 * 4 * EPS)


@pytest.mark.parametrize("unit", [2.0**-1000, 2.0**-665, 2.0**-530, 2.0**-515, 2.0**-100, 2.0**500, 2.0**515, 2.0**1000])
def test_symeig_norms(lanes_lib, unit):
    """An ordinary matrix at the ends of the range of a double."""
    A = np.random.default_rng(8).standard_normal((20, 20))
    _check_eigh(lanes_lib, A + A.T, 1e-12, unit)


@pytest.mark.parametrize("solver", ["host_symeig", "host_symeig_lds"])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_symeig_slots_stay_a_permutation(lanes_lib, solver, value):
    """A matrix with a NaN or infinite entry: no eigenvalues, but the columns' order still names every slot
    once (a slot left out would be read from whatever the LDS held).  The order alone is looked at: symeig_lds.h's
    numbers rely on a wave's lanes reading a row together before one of them changes it, which fibers do not."""
    rng = np.random.default_rng(2)
    for n, at in ((5, (1, 1)), (12, (7, 2)), (24, (0, 0))):
        A = rng.standard_normal((n, n))
        A = A + A.T
        A[at] = A[at[::-1]] = value
        perm = _eigh(lanes_lib, A, solver=solver)[2]
        assert sorted(perm) == list(range(n))


@pytest.mark.parametrize("B,N", [(1, 5), (32, 513), (2093062, 513), (2093063, 513), (4186128, 513), (2**31 - 1, 1024)])
def test_launches_cover_the_batch(lanes_lib, B, N):
    """The launches of a network adjoint: every system once, in order, and no point number past 2^31 even in the
    tiles past the end that the last round addresses (256 workgroups of 2 groups of 32 points)."""
    first, n = np.zeros(4096, dtype=np.int32), np.zeros(4096, dtype=np.int32)
    k = lanes_lib.host_launches(B, N, len(n), _p(first), _p(n))
    assert 1 <= k <= len(n)
    assert k == 1 or B * N > 2**30
    ends = np.cumsum(n[:k].astype(np.int64))
    assert ends[-1] == B and first[0] == 0 and (n[:k] > 0).all()
    assert (first[1:k] == ends[:-1]).all()
    assert n[:k].max() * N + 2 * 256 * 2 * 32 < 2**31
