"""The current where its G-space moments come from the sweeps: cubic and rectangular
grids, planes of each workgroup size (20 x 20 to 96 x 96), one band and several,
one band chunk and two, against the CPU oracle.

Tolerance 1e-12 relative to the norm of the current's own terms, as for the
current on other grids.
"""
import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from inq_amd import systems

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("n,nst,chunk", [
    ((20, 20, 20), 1, 0), ((20, 25, 24), 11, 8), ((24, 24, 24), 9, 0),
    ((36, 32, 27), 5, 0), ((48, 48, 48), 4, 0), ((72, 75, 20), 3, 0),
    ((96, 96, 20), 2, 0), ((80, 80, 80), 2, 0), ((60, 64, 24), 5, 0), ((64, 64, 64), 3, 0),
])
def test_current(device, n, nst, chunk):
    print("[gpu-test] current", n, nst, chunk, flush=True)
    lat = np.diag([0.4 * m for m in n])
    s = systems.make_system(n, lat, np.array([[1.0, 1.2, 0.8], [4.0, 3.0, 5.0]]), seed=5,
                            system_id=nst)
    rng = np.random.default_rng(nst)
    psi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    kA = (0.05, -0.04, 0.03)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    if chunk:
        ham.tuning = {"band_chunk": chunk}
    ham.uniform_vector_potential = kA
    _, got = ham.current(torch.from_numpy(psi).to(device), occ=2.0)
    _, ref = O.System(s.n, s.lattice, s.vloc, s.tables).current(psi, kA, 2.0, commutator="inq")
    scale = 2.0 * np.linalg.norm(psi) ** 2 * abs(np.linalg.det(lat)) / np.prod(n)
    assert np.abs(np.asarray(got) - ref).max() < TOL * max(scale, np.abs(ref).max())
    ham.close()


@pytest.mark.parametrize("n", [(24, 24, 24), (20, 25, 24)])
def test_bits_do_not_depend_on_the_chunk(device, n):
    """256 bands in rows of 256: one chunk, and chunks of interleaved groups of
    eight bands."""
    nst = 256
    print("[gpu-test] current chunks", n, flush=True)
    lat = np.diag([0.4 * m for m in n])
    s = systems.make_system(n, lat, np.array([[1.0, 1.2, 0.8], [4.0, 3.0, 5.0]]), seed=5,
                            system_id=nst)
    rng = np.random.default_rng(nst)
    psi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    d = torch.from_numpy(psi).to(device)
    kA = (0.05, -0.04, 0.03)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst, tuning=None)
    ham.uniform_vector_potential = kA
    _, got = ham.current(d, occ=2.0)
    _, ref = O.System(s.n, s.lattice, s.vloc, s.tables).current(psi, kA, 2.0, commutator="inq")
    scale = 2.0 * np.linalg.norm(psi) ** 2 * abs(np.linalg.det(lat)) / np.prod(n)
    assert np.abs(np.asarray(got) - ref).max() < TOL * max(scale, np.abs(ref).max())
    for chunk in (64, 128, 32):
        ham.tuning = {"band_chunk": chunk}
        assert np.array_equal(np.asarray(ham.current(d, occ=2.0)[1]), np.asarray(got)), chunk
    ham.close()
