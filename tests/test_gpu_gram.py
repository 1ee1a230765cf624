"""The inner products of the eigensolver at the edges of their tiles (16 bands) and
blocks (64 bands), on grids that leave a short last slice, allow a few or only
one, in both uses: the overlap matrix of orthogonalize against the CPU oracle, and the
subspace Hamiltonian by its eigenvalues against numpy's of the same matrix.

Tolerance 1e-12 relative: sums over up to 5e4 points in another order, times a
condition number below 10 for random bands.
"""
import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from helpers import relerr
from inq_amd import ground_state, systems

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("n,nst", [((12, 10, 14), 1), ((12, 10, 14), 16), ((12, 11, 10), 17),
                                   ((24, 24, 24), 33), ((32, 27, 25), 48), ((24, 25, 20), 49),
                                   ((12, 11, 10), 64), ((32, 27, 25), 65), ((36, 36, 36), 97),
                                   ((36, 36, 36), 130), ((12, 12, 12), 60), ((8, 10, 9), 97)])
def test_inner_products(device, n, nst):
    print("[gpu-test] gram", n, nst, flush=True)
    lat = np.diag([0.4 * m for m in n])
    s = systems.make_system(n, lat, np.zeros((0, 3)), with_projectors=False)
    rng = np.random.default_rng(nst)
    phi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst + 3)
    got = ground_state.orthogonalize(ham, torch.from_numpy(phi).to(device)).cpu().numpy()
    flat = phi.reshape(-1, nst)
    dV = abs(np.linalg.det(lat)) / flat.shape[0]
    assert relerr(got, O.orthogonalize(phi, dV)) < TOL

    hphi = ham(torch.from_numpy(phi).to(device)).cpu().numpy().reshape(-1, nst)
    ref = np.linalg.eigvalsh(dV * (flat.conj().T @ hphi))
    eig = ground_state.subspace_diagonalization(ham, torch.from_numpy(phi).to(device))
    assert np.abs(eig - ref).max() < TOL * np.abs(ref).max()
    ham.close()
