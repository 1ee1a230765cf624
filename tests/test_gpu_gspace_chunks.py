"""The G-space sweeps on band chunks of every size: a band's bits do not depend on
the chunk it falls in, with the projector's point sums split over workgroups or
not, where a chunk's partial sums take several launches, and where the chunks are
interleaved groups of eight bands (rows of 256 or 512 bands), as for steepest
descent with its preconditioner and line sums; G-space Hpsi of every cubic length;
V_nl psi kept per ownership entry (nine channels) on a grid of the rectangular
sweeps.

Tolerances against the CPU oracle 1e-12 relative; steepest descent 1e-10, whose five
line searches amplify the last bits.
"""
import ctypes

import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from helpers import relerr
from inq_amd import ground_state, operations, systems

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


@pytest.mark.parametrize("n", [(24, 24, 24), (20, 25, 24)])
def test_descent_on_band_groups(device, n):
    """256 bands in one chunk and in chunks of interleaved groups, with and without
    the preconditioner."""
    nst = 256
    print("[gpu-test] descent groups", n, flush=True)
    lat = np.diag([0.4 * m for m in n])
    s = systems.make_system(n, lat, np.array([[1.0, 1.2, 0.8], [4.0, 3.0, 5.0]]), seed=3)
    phi = systems.random_orbitals(s, nst, ecut=15.0, fourier=True)
    osys = O.System(s.n, s.lattice, s.vloc, s.tables)
    d = torch.from_numpy(phi).to(device)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst, tuning=None)
    hphi = ham(d, fourier=True)
    assert relerr(hphi.cpu().numpy(), osys.hamiltonian_fourier(phi)) < TOL
    for pre in (True, False):
        ham.tuning = {"band_chunk": 0}
        one = ground_state.steepest_descent(ham, d.clone(), precondition=pre)
        if pre:
            assert relerr(one.cpu().numpy(), osys.steepest_descent(phi)) < 1e-10
        for chunk in (64, 128, 48):
            ham.tuning = {"band_chunk": chunk}
            assert torch.equal(ham(d, fourier=True), hphi), chunk
            got = ground_state.steepest_descent(ham, d.clone(), precondition=pre)
            assert torch.equal(got, one), (pre, chunk)
    ham.close()


@pytest.mark.parametrize("n", [(24, 24, 24), (20, 25, 24)])
def test_ragged_band_groups(device, n):
    """264 bands in rows of 512: 33 groups over five chunks, in real space and in G
    space, against rows of 264 (contiguous chunks)."""
    nst = 264
    print("[gpu-test] ragged groups", n, flush=True)
    lat = np.diag([0.4 * m for m in n])
    s = systems.make_system(n, lat, np.array([[1.0, 1.2, 0.8], [4.0, 3.0, 5.0]]), seed=3)
    g = torch.Generator(device=device).manual_seed(5)
    src = torch.randn(n + (nst,), dtype=torch.complex128, device=device, generator=g)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst, tuning=None)
    ham.uniform_vector_potential = kA = (0.05, -0.04, 0.03)
    ham.tuning = {"band_chunk": 56}
    osys = O.System(s.n, s.lattice, s.vloc, s.tables)
    host = np.ascontiguousarray(src[..., [0, 100, 263]].cpu().numpy())
    for name, exact in (("inqamd_hamiltonian_apply", osys.hamiltonian(host, kA)),
                        ("inqamd_hamiltonian_apply_fourier", osys.hamiltonian_fourier(host, kA))):
        outs = []
        for ld in (512, 264):
            a = torch.zeros(n + (ld,), dtype=torch.complex128, device=device)
            a[..., :nst] = src
            o = torch.zeros_like(a)
            torch.cuda.synchronize()
            ham.handle.call(name, ctypes.c_void_p(a.data_ptr()), ctypes.c_void_p(o.data_ptr()), nst,
                            ld)
            torch.cuda.synchronize()
            assert torch.count_nonzero(o[..., nst:]).item() == 0
            outs.append(o[..., :nst])
        assert torch.equal(outs[0], outs[1]), name
        assert relerr(outs[0][..., [0, 100, 263]].cpu().numpy(), exact) < TOL
    J = []
    for ld in (512, 264):
        a = torch.zeros(n + (ld,), dtype=torch.complex128, device=device)
        a[..., :nst] = src
        torch.cuda.synchronize()
        cov, cart = (ctypes.c_double * 3)(), (ctypes.c_double * 3)()
        ham.handle.call("inqamd_current", ctypes.c_void_p(a.data_ptr()), nst, ld,
                        ctypes.c_double(2.0), cov, cart)
        J.append(list(cart))
    assert J[0] == J[1]
    ham.close()


@pytest.mark.parametrize("length", [24, 30, 32, 36, 40, 48, 60, 64, 72, 80, 96])
def test_every_cubic_length(device, length):
    n, nst = (length,) * 3, 3
    print("[gpu-test] G-space", n, flush=True)
    lat = np.diag([0.4 * m for m in n])
    atoms = np.array([[1.0, 1.2, 0.8], [4.0, 3.0, 5.0], [7.0, 7.5, 2.0]])
    s = systems.make_system(n, lat, atoms, seed=3, system_id=length)
    rng = np.random.default_rng(length)
    phi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    ham.uniform_vector_potential = kA = (0.05, -0.04, 0.03)
    got = ham(torch.from_numpy(phi).to(device), fourier=True).cpu().numpy()
    ref = O.System(s.n, s.lattice, s.vloc, s.tables).hamiltonian_fourier(phi, kA)
    assert relerr(got, ref) < TOL
    ham.close()


def test_nine_channels_on_a_rectangular_grid(device):
    n, nst, nlm = (25, 36, 27), 11, 9
    lat = np.diag([0.4 * m for m in n])
    rng = np.random.default_rng(9)
    s = systems.make_system(n, lat, np.zeros((0, 3)), with_projectors=False)
    s.vloc = rng.standard_normal(n)
    s.atoms = rng.uniform(0.0, 1.0, (3, 3)) @ lat
    t = systems.projector_tables(lat, n, s.atoms, 1.8, 0.9, 4, np.zeros((3, 4)))
    t.update(max_nlm=nlm, nlm=np.full(3, nlm, np.int32), coeff=rng.uniform(-1, 1, (3, nlm)),
             matrices=rng.standard_normal((3, nlm, t["max_sphere"])))
    s.tables = t
    psi = rng.standard_normal(n + (nst,)) + 1j * rng.standard_normal(n + (nst,))
    osys = O.System(s.n, s.lattice, s.vloc, s.tables)
    ham = inq_amd.ks_hamiltonian(s, max_bands=nst)
    ham.uniform_vector_potential = kA = (0.05, -0.04, 0.03)
    d = torch.from_numpy(psi).to(device)
    assert relerr(ham(d).cpu().numpy(), osys.hamiltonian(psi, kA)) < TOL
    assert relerr(ham(d, fourier=True).cpu().numpy(), osys.hamiltonian_fourier(psi, kA)) < TOL
    got = operations.exponential_in_place(ham, 0.01j, d.clone(), 4).cpu().numpy()
    assert relerr(got, osys.exponential_in_place(psi, 0.01j, 4, kA)) < TOL
    ham.close()
