"""The in-place rotations of the eigensolver at the edges of their forms (64 bands per
workgroup of four row tiles; 316 with 32 rows in LDS, 636 with 16, a library
product beyond), with a last workgroup cut short: upper triangular in
orthogonalize against the CPU oracle, full in the subspace diagonalisation, whose
orbitals must diagonalise H with the eigenvalues that it returns.

Tolerance 1e-11 relative: products of up to 637 terms with random bands whose overlap
matrix has a condition number up to about 20 (637 bands on 1680 points).
"""
import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from helpers import relerr
from inq_amd import ground_state, systems

pytestmark = pytest.mark.gpu
TOL = 1e-11


@pytest.mark.parametrize("nst", [3, 63, 64, 65, 130, 316, 317, 636, 637])
def test_rotations(device, nst):
    n = (12, 10, 14)
    print("[gpu-test] rotate", n, nst, flush=True)
    lat = np.diag([0.4 * m for m in n])
    s = systems.make_system(n, lat, np.zeros((0, 3)), with_projectors=False)
    rng = np.random.default_rng(nst)
    phi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    dV = abs(np.linalg.det(lat)) / np.prod(n)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    got = ground_state.orthogonalize(ham, torch.from_numpy(phi).to(device)).cpu().numpy()
    assert relerr(got, O.orthogonalize(phi, dV)) < TOL

    d = torch.from_numpy(phi).to(device)
    eig = ground_state.subspace_diagonalization(ham, d)
    out, hout = d.cpu().numpy().reshape(-1, nst), ham(d).cpu().numpy().reshape(-1, nst)
    sub = dV * (out.conj().T @ hout)
    assert np.abs(sub - np.diag(eig)).max() < TOL * np.abs(eig).max()
    assert abs(np.linalg.norm(out) / np.linalg.norm(phi) - 1) < TOL
    ham.close()
