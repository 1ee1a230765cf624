"""Taylor sums of every order around the four terms that one sweep adds (fewer
pending powers, exactly three, several groups, a last group of one) against the
CPU oracle: in place, as a copy and 2-for-1, with and without projectors, on the
smallest three-sweep grid and on a pencil grid.

Tolerance 1e-12 relative 2-norm, as for the other propagator tests.
"""
import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from helpers import relerr
from inq_amd import operations, systems

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5, 7, 8, 9])
@pytest.mark.parametrize("n,nst,natoms", [((24, 24, 24), 9, 3), ((24, 24, 24), 3, 0),
                                          ((12, 11, 10), 5, 2)])
def test_orders(device, order, n, nst, natoms):
    print("[gpu-test] taylor order", order, n, nst, natoms, flush=True)
    lat = np.diag([0.4 * m for m in n])
    rng = np.random.default_rng(order)
    s = systems.make_system(n, lat, rng.uniform(0, 1, (natoms, 3)) @ lat, seed=2, system_id=7)
    psi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    kA = (0.03, 0.02, -0.05)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    ham.uniform_vector_potential = kA
    osys = O.System(s.n, s.lattice, s.vloc, s.tables)
    z1, z2 = 0.01j, 0.02j
    d = torch.from_numpy(psi).to(device)
    ref1 = osys.exponential_in_place(psi, z1, order, kA)
    got = operations.exponential_in_place(ham, z1, d.clone(), order)
    assert relerr(got.cpu().numpy(), ref1) < TOL
    phi = d.clone()
    exp = operations.exponential_2_for_1(ham, z1, z2, phi, order)
    assert relerr(exp.cpu().numpy(), ref1) < TOL
    assert relerr(phi.cpu().numpy(), osys.exponential_in_place(psi, z2, order, kA)) < TOL
    ham.close()
