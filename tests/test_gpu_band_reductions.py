"""The per-band reductions of the eigensolver in each of their shapes (16 and 64
bands per block, full and ragged groups; chunks of the shortest and of the full
length and one in between, the last one cut short) against the CPU oracle.

Tolerance 1e-12 relative 2-norm, as for the other eigensolver tests.
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


@pytest.mark.parametrize("n,nst", [((12, 10, 14), 1), ((12, 10, 14), 16), ((12, 10, 14), 63),
                                   ((12, 11, 10), 64), ((12, 10, 14), 65), ((64, 64, 64), 3),
                                   ((72, 80, 90), 50), ((60, 60, 50), 17),
                                   ((50, 50, 54), 130)])
def test_preconditioner_shapes(device, n, nst):
    """operations::preconditioner: the kinetic sums and their use."""
    print("[gpu-test] reductions", n, nst, flush=True)
    lat = np.diag([0.4 * m for m in n])
    s = systems.make_system(n, lat, np.zeros((0, 3)), with_projectors=False)
    rng = np.random.default_rng(nst)
    phi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    got = ground_state.preconditioner(ham, torch.from_numpy(phi).to(device)).cpu().numpy()
    ref = O.System(s.n, s.lattice, s.vloc, s.tables).preconditioner(phi)
    assert relerr(got, ref) < TOL
    ham.close()


@pytest.mark.parametrize("nst", [5, 20, 64, 70])
def test_descent_shapes(device, nst):
    n = (12, 10, 14)
    lat = np.diag([0.5 * m for m in n])
    s = systems.make_system(n, lat, np.array([[1.0, 1.2, 0.8], [4.0, 3.0, 5.0]]), seed=3,
                            system_id=nst)
    phi = systems.random_orbitals(s, nst, ecut=15.0, fourier=True)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    got = ground_state.steepest_descent(ham, torch.from_numpy(phi).to(device)).cpu().numpy()
    ref = O.System(s.n, s.lattice, s.vloc, s.tables).steepest_descent(phi)
    assert relerr(got, ref) < 1e-10  # five line searches amplify the last bits
    ham.close()
