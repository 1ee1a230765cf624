"""The three-sweep Hpsi on nx x ny x nz grids against the CPU oracle: every
length on every axis, planes of every workgroup size, ragged band tiles and
band chunks, with V_nl psi from the coefficients, in real space and in G space;
the Taylor chains and the adjoint's fused half steps on such a grid; cubic grids
of the lengths that have no cubic kernels.

Tolerance 1e-12 relative 2-norm (the adjoint 1e-9 against the form that stores
no powers, whose sums are formed in another order).
"""
import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from helpers import relerr
from inq_amd import adjoint, operations, systems

pytestmark = pytest.mark.gpu
TOL = 1e-12
LENGTHS = (20, 24, 25, 27, 28, 30, 32, 36, 40, 42, 45, 48, 50, 54, 56, 60, 64, 70, 72, 75, 80, 84,
           90, 96)


def make(n, nst, natoms, seed=1):
    lat = np.diag([0.4 * m for m in n])
    if natoms:  # a cell that is not orthorhombic
        lat[1, 0], lat[2, 1] = 1.0, -0.5
    rng = np.random.default_rng(seed + nst)
    s = systems.make_system(n, np.diag(np.diag(lat)), np.zeros((0, 3)), with_projectors=False)
    s.lattice = lat
    s.vloc = rng.standard_normal(n)
    if natoms:
        s.atoms = rng.uniform(0, 1, (natoms, 3)) @ lat
        s.tables = systems.projector_tables(lat, n, s.atoms, 1.8, 0.9, 4,
                                            rng.uniform(-1, 1, (natoms, 4)))
    psi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    return s, psi, O.System(s.n, s.lattice, s.vloc, s.tables)


def check(device, n, nst, natoms):
    print("[gpu-test] rect", n, nst, natoms, flush=True)
    s, psi, osys = make(n, nst, natoms)
    kA = (0.05, -0.04, 0.03)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    ham.uniform_vector_potential = kA
    d = torch.from_numpy(psi).to(device)
    assert relerr(ham(d).cpu().numpy(), osys.hamiltonian(psi, kA)) < TOL
    return s, psi, osys, ham, d, kA


@pytest.mark.parametrize("length", LENGTHS)
def test_every_length_on_every_axis(device, length):
    for n, nst in (((length, 20, 24), 2), ((24, length, 20), 3), ((20, 24, length), 1)):
        check(device, n, nst, 0)[3].close()


@pytest.mark.parametrize("n,nst,natoms", [
    ((96, 96, 20), 3, 2), ((64, 90, 25), 9, 3), ((48, 50, 36), 17, 4), ((24, 27, 80), 8, 3),
    ((25, 25, 25), 11, 2), ((90, 90, 90), 2, 0), ((20, 20, 20), 5, 1),
    ((60, 64, 20), 3, 0), ((72, 70, 24), 5, 0), ((60, 64, 20), 9, 3), ((72, 70, 24), 3, 2),
])
def test_hpsi_gspace_and_etrs(device, n, nst, natoms):
    s, psi, osys, ham, d, kA = check(device, n, nst, natoms)
    got = ham(d, fourier=True).cpu().numpy()
    assert relerr(got, osys.hamiltonian_fourier(psi, kA)) < TOL
    z = 0.01j
    ref = osys.exponential_in_place(psi, z, 4, kA)
    got = operations.exponential_in_place(ham, z, d.clone(), 4).cpu().numpy()
    assert relerr(got, ref) < TOL
    ham.close()


def test_band_chunks(device):
    """Several band chunks on two streams: each band's bits do not depend on
    the chunk it falls in."""
    n, nst = (30, 36, 40), 20
    s, psi, osys, ham, d, kA = check(device, n, nst, 3)
    one = ham(d).clone()
    ham.tuning = {"band_chunk": 8}
    assert torch.equal(ham(d), one)
    ham.close()


def test_adjoint_gradients(device):
    """The fused half steps against the form that recomputes the powers."""
    n, nst = (20, 27, 24), 5
    s, psi, _ = make(n, nst, 2)
    d = torch.from_numpy(psi / np.linalg.norm(psi)).to(device)
    coef = np.array([0.05, -0.03, 0.02])
    out = []
    for store in (True, False):
        ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
        prop = adjoint.propagation_adjoint(ham, nst, nsteps=4, dt=0.02, ncoef=3, omega=0.3,
                                           checkpoint_every=2, store_powers=store)
        loss, _ = prop.forward(coef, d)
        gc, gV, lam = prop.backward(1.0, want_lambda0=True)
        out.append((loss, np.array(gc), gV.cpu().numpy(), lam.cpu().numpy()))
        prop.close()
        ham.close()
    assert abs(out[0][0] - out[1][0]) <= 1e-12 * abs(out[1][0])
    for a, b in zip(out[0][1:], out[1][1:]):
        assert relerr(a, b) < 1e-9
