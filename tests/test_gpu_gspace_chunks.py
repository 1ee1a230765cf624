"""G-space Hpsi on band chunks of every size: a band's bits do not depend on the
chunk it falls in, with the projector's point sums split over workgroups or not,
and where a chunk's partial sums take several launches.
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


@pytest.mark.parametrize("n,nst,natoms,chunks", [
    # 64 spheres: a chunk of 32 bands alone would split their points, all bands not
    ((32, 32, 32), 80, 64, (32, 64, 8)),
    # the same on a grid of the rectangular sweeps, with a short last chunk
    ((36, 30, 32), 74, 64, (32, 64)),
    # 120 spheres: the split of the library's 32-band chunk, more bands than the
    # partial sums of one launch hold
    ((72, 72, 72), 144, 120, (144, 24)),
])
def test_bits_do_not_depend_on_the_chunk(device, n, nst, natoms, chunks):
    print("[gpu-test] G-space chunks", n, nst, natoms, flush=True)
    lat = np.diag([float(m) for m in n]) * (10.26 / 32)
    atoms = np.random.default_rng(natoms).uniform(0.0, 1.0, (natoms, 3)) @ lat
    s = systems.make_system(n, lat, atoms, seed=3, system_id=natoms)
    assert s.tables["max_sphere"] >= 512  # two chunks of points
    g = torch.Generator(device=device).manual_seed(nst)
    phi = torch.randn(n + (nst,), dtype=torch.complex128, device=device, generator=g)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst, tuning=None)
    ham.uniform_vector_potential = kA = (0.05, -0.04, 0.03)
    ref = ham(phi, fourier=True)
    few = [0, nst - 1]
    host = np.ascontiguousarray(phi[..., few].cpu().numpy())
    exact = O.System(s.n, s.lattice, s.vloc, s.tables).hamiltonian_fourier(host, kA)
    assert relerr(ref[..., few].cpu().numpy(), exact) < TOL
    for chunk in chunks:
        ham.tuning = {"band_chunk": chunk}
        assert torch.equal(ham(phi, fourier=True), ref), chunk
    ham.close()
