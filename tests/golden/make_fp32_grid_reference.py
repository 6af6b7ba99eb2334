"""Density matrices of 16-atom chains from the FP32 grid path of the 3D SCF (needs the GPU).

The chain of ``synthetic_chain(16, 116)`` (80 functions) with its bonds displaced by up to 0.2 %; of 72
such chains these five moved by 2e-9 .. 8e-9 when another FP64 eigensolver and order of sums ran
the cycles.  Written by the library of commit 06972af, whose order of operations the path keeps; stored are
the geometry, the shells, the energy and the density matrix's diagonal.
Writes fp32_grid_chains.npz beside this script.

    python tests/golden/make_fp32_grid_reference.py
"""

import os
import sys

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
sys.path.insert(0, ROOT)

# (seed, chains of 16, 8, 4 and 2 atoms drawn before it)
CHAINS = ((1, 16), (6, 12), (8, 0), (9, 16), (11, 4))
BOHR = 0.52917721092


def chain(seed, skip):
    rng = np.random.default_rng([seed, 2])
    for k in range(skip):
        rng.uniform(0.998, 1.002, (16, 8, 4, 2)[k % 4] - 1)
    base = np.random.default_rng(116)
    bonds = base.uniform(0.5, 1.5, 15) / BOHR * rng.uniform(0.998, 1.002, 15)
    exps, coefs = np.zeros((16, 3, 3)), np.zeros((16, 3, 3))
    for a in range(16):
        for s in range(3):
            exps[a, s] = np.sort(np.exp(base.uniform(np.log(0.1), np.log(20.0), 3)))[::-1]
            coefs[a, s] = base.uniform(0.2, 1.0, 3)
    z = np.concatenate([[0.0], np.cumsum(bonds)])
    return z - z.mean(), exps, coefs


def solve(td, zs, exps, coefs):
    """The SCF of the chains with atoms at zs (bohr), as one batch."""
    shells = [[(l, exps[a, s], coefs[a, s]) for s, l in enumerate((0, 0, 1))] for a in range(16)]
    mfs = []
    for z in zs:
        mol = td.gto.Mole([("H", (0.0, 0.0, x)) for x in z], basis="6-31g", unit="Bohr", shells_per_atom=shells)
        mf = td.scf.RKS(mol)
        mf.conv_tol, mf.max_cycle, mf.diis_space, mf.precision = 1e-8, 30, 8, "fp32_grid"
        mfs.append(mf)
    e = td.scf.kernel_batch(mfs)
    return np.array(e), np.stack([mf.dm.diagonal().cpu().numpy() for mf in mfs])


def main():
    from qex_amd import td

    data = [chain(*c) for c in CHAINS]
    zs = np.stack([d[0] for d in data])
    e, diag = solve(td, zs, data[0][1], data[0][2])
    path = os.path.join(HERE, "fp32_grid_chains.npz")
    np.savez(path, z=zs, exps=data[0][1], coefs=data[0][2], e_tot=e, dm_diag=diag)
    print(path, e, np.abs(diag).max())


if __name__ == "__main__":
    main()
