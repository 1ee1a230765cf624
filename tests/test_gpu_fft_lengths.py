"""Pencil passes over every axis length and over ragged column counts against
the CPU oracle: lengths with a butterfly plan, lengths that go through the DFT
matrix (primes, prime multiples, the shortest and the longest of its range, one
beyond it), each on every axis, in the transforms and in the kinetic and V psi
passes of H psi.

Tolerance 1e-12 relative 2-norm, as for the other transforms.
"""
import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from helpers import relerr
from inq_amd import systems
from inq_amd.operations import transform

pytestmark = pytest.mark.gpu
TOL = 1e-12

PLANNED = (8, 9, 10, 12, 14, 15, 16, 18, 20, 21, 24, 25, 27, 28, 30, 32, 35, 36, 40, 42, 45, 48,
           49, 50, 54, 56, 60, 63, 64, 70, 72, 75, 80, 81, 84, 90, 96, 100, 108, 112, 120, 125,
           126, 128)


def check(device, n, nst):
    print("[gpu-test] lengths", n, nst, flush=True)
    rng = np.random.default_rng(sum(n) + nst)
    lat = np.diag([0.4 * m for m in n])
    s = systems.make_system(n, lat, np.zeros((0, 3)), with_projectors=False)
    s.vloc[...] = rng.standard_normal(n)
    psi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    kA = (0.1, -0.2, 0.05)
    ham.uniform_vector_potential = kA
    d = torch.from_numpy(psi).to(device)
    f = transform.to_fourier(d, ham)
    assert relerr(f.cpu().numpy(), O.to_fourier(psi)) < TOL
    assert relerr(transform.to_real(f, ham, out=f).cpu().numpy(), psi) < TOL  # in place
    ref = O.System(s.n, s.lattice, s.vloc, s.tables).hamiltonian(psi, kA)
    assert relerr(ham(d).cpu().numpy(), ref) < TOL
    ham.close()


@pytest.mark.parametrize("length", PLANNED)
def test_planned_length(device, length):
    check(device, (length, 5, length) if length < 64 else (3, 4, length), 3)
    check(device, (4, length, 3), 17)


@pytest.mark.parametrize("length", [1, 2, 3, 4, 5, 6, 7, 11, 13, 17, 29, 31, 32 + 1, 37, 44, 47, 52,
                                    62, 67, 94, 95, 97, 127, 131, 133, 190, 191])
def test_dft_matrix_length(device, length):
    check(device, (length, 5, length) if length < 48 else (3, 2, length), 3)
    check(device, (3, length, 2), 16)
    check(device, (length, 2, 3), 1)


@pytest.mark.parametrize("length", [144, 160, 192, 194])
def test_beyond_both(device, length):
    check(device, (2, length, 3), 9)
