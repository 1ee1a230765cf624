"""Steepest descent on grids whose last G-space sweep also forms the line
search's sums, against the CPU oracle: ragged band tiles (1, 5, 17, 20 bands in
tiles of 8), ragged row tiles (25 to 30 rows in tiles of 8), cubic and rectangular
grids, one band chunk and several.

Tolerance 1e-10 relative 2-norm: the operator holds 1e-12, and five line searches
amplify the last bits.
"""
import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from helpers import relerr
from inq_amd import ground_state, systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nst,chunk", [
    ((24, 24, 24), 1, 0), ((24, 24, 24), 17, 0), ((24, 24, 24), 20, 8), ((36, 36, 36), 5, 0),
    ((20, 25, 24), 17, 8), ((28, 30, 36), 5, 0), ((32, 27, 25), 8, 0),
])
def test_descent(device, n, nst, chunk):
    print("[gpu-test] line search", n, nst, chunk, flush=True)
    lat = np.diag([0.5 * m for m in n])
    s = systems.make_system(n, lat, np.array([[1.0, 1.2, 0.8], [4.0, 3.0, 5.0]]), seed=3,
                            system_id=nst)
    phi = systems.random_orbitals(s, nst, ecut=15.0, fourier=True)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    if chunk:
        ham.tuning = {"band_chunk": chunk}
    ref = O.System(s.n, s.lattice, s.vloc, s.tables).steepest_descent(phi)
    got = ground_state.steepest_descent(ham, torch.from_numpy(phi).to(device)).cpu().numpy()
    assert relerr(got, ref) < 1e-10
    ham.close()
