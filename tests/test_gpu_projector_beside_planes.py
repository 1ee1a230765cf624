"""The projector's coefficients and phases computed by workgroups of the sweeps'
own launches, at the edges of the rule that takes them there (plane counts and
(sphere, band tile) counts on either side of its limits, one band, ragged band
tiles, one and several band chunks), against the CPU oracle.

Tolerance 1e-12 relative 2-norm.
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


@pytest.mark.parametrize("n,nst,natoms,chunk", [
    ((24, 24, 24), 1, 1, 0), ((24, 24, 24), 17, 3, 8), ((32, 32, 32), 64, 2, 0),
    ((32, 32, 32), 65, 2, 0), ((48, 48, 48), 33, 2, 16), ((24, 24, 24), 16, 511, 0),
    ((24, 24, 24), 16, 512, 0), ((20, 27, 24), 18, 3, 8), ((64, 54, 20), 5, 4, 0),
    ((96, 60, 20), 3, 4, 0),
])
def test_hpsi_and_taylor(device, n, nst, natoms, chunk):
    print("[gpu-test] projector beside planes", n, nst, natoms, chunk, flush=True)
    lat = np.diag([0.4 * m for m in n])
    rng = np.random.default_rng(nst + natoms)
    s = systems.make_system(n, lat, rng.uniform(0, 1, (min(natoms, 8), 3)) @ lat, seed=4, system_id=1)
    if natoms > 8:  # many small spheres
        s.tables = systems.projector_tables(lat, n, rng.uniform(0, 1, (natoms, 3)) @ lat, 0.9, 0.5, 4,
                                            rng.uniform(-1, 1, (natoms, 4)))
    psi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    kA = (0.04, -0.03, 0.02)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    ham.uniform_vector_potential = kA
    if chunk:
        ham.tuning = {"band_chunk": chunk}
    osys = O.System(s.n, s.lattice, s.vloc, s.tables)
    d = torch.from_numpy(psi).to(device)
    assert relerr(ham(d).cpu().numpy(), osys.hamiltonian(psi, kA)) < TOL
    # another vector potential on the same handle: the phases are the call's
    kB = (-0.05, 0.01, 0.06)
    ham.uniform_vector_potential = kB
    got = operations.exponential_in_place(ham, 0.01j, d.clone(), 2).cpu().numpy()
    assert relerr(got, osys.exponential_in_place(psi, 0.01j, 2, kB)) < TOL
    ham.close()
