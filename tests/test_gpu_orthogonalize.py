"""The device Cholesky factorisation behind orthogonalize, around its blocks of
32 and strips of 8 (one band, one under and over a block, several blocks, a
ragged last one): against the oracle's Gram-Schmidt, by the orthonormality of
the result, and the refusal of an overlap without a factor.

Tolerance 1e-12 relative 2-norm against the oracle and 1e-12 on the overlap (the
overlaps here are well conditioned).
"""
import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from helpers import relerr
from inq_amd import _lib, ground_state, systems

pytestmark = pytest.mark.gpu
TOL = 1e-12


def handle(nst):
    n = (12, 10, 14)
    s = systems.make_system(n, np.diag([5.0, 4.5, 6.0]), np.zeros((0, 3)), with_projectors=False)
    return s, inq_amd.ks_hamiltonian(s, max_bands=nst)


@pytest.mark.parametrize("nst", [1, 7, 31, 32, 33, 64, 65, 100, 200])
def test_orthogonalize_blocks(device, nst):
    print("[gpu-test] orthogonalize", nst, flush=True)
    s, ham = handle(nst)
    rng = np.random.default_rng(nst)
    phi = rng.standard_normal(s.n + (nst,)) + 1j * rng.standard_normal(s.n + (nst,))
    dV = s.volume / s.npoints
    d = ground_state.orthogonalize(ham, torch.from_numpy(phi).to(device))
    got = d.cpu().numpy().reshape(-1, nst)
    assert relerr(got, O.orthogonalize(phi, dV).reshape(-1, nst)) < TOL
    assert np.abs(dV * (got.conj().T @ got) - np.eye(nst)).max() < TOL
    ham.close()


@pytest.mark.parametrize("band", [0, 5, 40])
def test_no_factor_is_refused_and_keeps_phi(device, band):
    nst = 45
    s, ham = handle(nst)
    rng = np.random.default_rng(1)
    phi = rng.standard_normal(s.n + (nst,)) + 1j * rng.standard_normal(s.n + (nst,))
    phi[..., band] = 0.0
    d = torch.from_numpy(phi).to(device)
    with pytest.raises(_lib.InqAmdError, match=f"not positive definite \\(band {band}\\)"):
        ground_state.orthogonalize(ham, d)
    assert np.array_equal(d.cpu().numpy(), phi)
    ham.close()
