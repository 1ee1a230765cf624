"""The per-band energy terms over the shapes of their reductions against the
CPU oracle: band counts around the 8 bands of a totals workgroup and the 64 of
a partial-sum block, grids of fewer and of more point chunks than its 128
lanes, with and without projectors, and channels whose coefficient is zero.

Tolerance 1e-12 relative (2-norm over the bands), as for every reduction.
"""
import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from helpers import relerr
from inq_amd import systems

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("n,nst,natoms", [
    ((12, 10, 14), 1, 2), ((12, 10, 14), 9, 0), ((24, 24, 24), 8, 3), ((20, 24, 30), 65, 2),
    ((36, 36, 36), 7, 5),
])
def test_energy_terms(device, n, nst, natoms):
    print("[gpu-test] energy terms", n, nst, natoms, flush=True)
    lat = np.diag([m * 0.4 for m in n])
    rng = np.random.default_rng(nst)
    s = systems.make_system(n, lat, rng.uniform(0, 1, (natoms, 3)) @ lat, seed=5, system_id=nst)
    if natoms:
        s.tables["coeff"][0, 1] = 0.0
        s.tables["coeff"][-1, 3] = 0.0
    psi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    kA = (0.04, -0.03, 0.02)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    ham.uniform_vector_potential = kA
    got = [t.cpu().numpy() for t in ham.energy(torch.from_numpy(psi).to(device))]
    ref = O.System(s.n, s.lattice, s.vloc, s.tables).energy(psi, kA)
    assert relerr(got[0], ref[0]) < TOL
    assert relerr(got[1], ref[1]) < TOL
    if natoms:
        assert relerr(got[2], ref[2]) < TOL
    else:
        assert np.all(got[2] == 0.0)
    ham.close()
