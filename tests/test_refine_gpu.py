"""The eigenpairs of the pentadiagonal Hamiltonian from one wave's substructured solves
(band_wave.h): cold starts (one non-interacting solve) and warm starts (SCF iterations) against dense
eigensolutions, over grid sizes at the edges of the rows-per-lane classes, with degenerate wells."""

import numpy as np
import pytest
import torch

from oracle import od as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def od():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import qex_amd.od as od
    return od


@pytest.mark.parametrize("N", [5, 6, 9, 10, 11, 64, 129, 319, 320, 321, 322, 448, 449, 512, 513, 577, 960, 961, 1023, 1024])
def test_cold_pairs_match_dense(od, N):
    """A batch of potentials (harmonic, double well at several separations down to a splitting of rounding
    size, flat, deep and narrow) at each N: eigenvalues to 1e-9, residuals and orthogonality of the states."""
    x = np.linspace(-10.0, 10.0, N)
    dx = x[1] - x[0]
    well = lambda r: -2.0 * np.exp(-np.abs(x - r)) - 2.0 * np.exp(-np.abs(x + r))
    pots = np.stack([0.5 * x ** 2, well(0.5), well(3.0), well(6.0), well(9.0), np.zeros(N), -50.0 * np.exp(-4 * x ** 2),
                     np.cos(3 * x)])
    k = min(4, N - 1)
    ne = 2 * (k - 1) if k > 1 else 1
    r = od.engine.solve_noninteracting(pots, [ne] * len(pots), x, with_states=True, max_electrons=ne)
    H0 = O.get_kinetic_matrix(x)
    for b, v in enumerate(pots):
        H = H0 + np.diag(v)
        w = np.linalg.eigvalsh(H)
        got = r.eigenvalues[b].cpu().numpy()
        psi = r.wavefunctions[b].cpu().numpy() * np.sqrt(dx)
        kk = ne // 2 + 1
        scale = np.abs(np.diag(H)).max() + 4.0 / dx ** 2
        np.testing.assert_allclose(got[:kk], w[:kk], rtol=0, atol=1e-9 * max(1.0, np.abs(w[:kk]).max()) + 1e-13 * scale)
        np.testing.assert_allclose(psi[:kk] @ psi[:kk].T, np.eye(kk), atol=1e-8)
        assert np.abs(H @ psi[:kk].T - psi[:kk].T * got[:kk]).max() < 1e-8 * max(1.0, scale * 1e-3)


@pytest.mark.parametrize("N", [65, 129, 320, 321, 513, 1024])
def test_warm_pairs_match_oracle(od, N):
    """Ten LDA iterations (warm from the second on), 1 to 7 electrons, a stretched pair included (4 bohr: at 10
    the loop breaks the symmetry from rounding, and the oracle itself moves by 0.1 Ha under a density
    perturbed by 1e-13)."""
    x = np.linspace(-15.0, 15.0, N)
    mols = [(np.array([0.0]), np.array([2]), 1), (np.array([-0.7, 0.7]), np.array([1, 1]), 2),
            (np.array([-2.0, 2.0]), np.array([1, 1]), 2), (np.array([-2.0, 0.3, 1.9]), np.array([3, 1, 3]), 7)]
    n0 = np.stack([O.gaussian_initial_density(x, *m, weighted=True) for m in mols])
    prob = od.engine.Problem1D(x, [m[0] for m in mols], [m[1] for m in mols], [m[2] for m in mols],
                               od.utils.exponential_coulomb, od.xc.LDAExp(), 10, alpha=0.3, alpha_decay=1.0,
                               num_mixing_iterations=1, loop="scan")
    r = prob.run(n0)
    for b, (loc, z, ne) in enumerate(mols):
        ref = O.jit_kohn_sham(loc, z, ne, 10, x, O.LDAExp(), O.exponential_coulomb, n0[b], alpha=0.3, alpha_decay=1.0,
                              num_mixing_iterations=1)
        np.testing.assert_allclose(r.total_energy[b].cpu().numpy(), ref.total_energy, rtol=0, atol=1e-8)
        np.testing.assert_allclose(r.density[b].cpu().numpy(), ref.density, rtol=0, atol=1e-7)
