"""The fused field passes (Hartree, PBE and the Kohn-Sham update on one real
field) against the CPU oracle: odd and even lengths, primes, axes around the
16-row blocks of the DFT-matrix product and the 16-column tiles, one axis beyond
its longest length (the general path), every functional part and combination.

Tolerance 1e-12 of the largest value (smooth positive densities; the PBE
potential divides by powers of the density, whose smallest here is a tenth of
its mean).
"""
import numpy as np
import pytest
import torch

import inq_amd
import oracle as O
from inq_amd import systems, tddft

pytestmark = pytest.mark.gpu
TOL = 1e-12


def density(n, seed=1):
    """A mean and a few long waves: positive, smooth on every axis."""
    x = np.meshgrid(*[2 * np.pi * np.arange(m) / m for m in n], indexing="ij")
    rng = np.random.default_rng(seed)
    rho = np.full(n, 0.2)
    for _ in range(4):
        k = rng.integers(-2, 3, 3)
        rho += 0.04 * np.cos(k[0] * x[0] + k[1] * x[1] + k[2] * x[2] + rng.uniform(0, 6.28))
    return rho


def close(a, b):
    return np.abs(np.asarray(a) - np.asarray(b)).max() <= TOL * np.abs(np.asarray(b)).max()


@pytest.mark.parametrize("n", [(20, 21, 22), (13, 7, 30), (31, 32, 33), (64, 5, 3), (6, 97, 8),
                               (8, 6, 131), (191, 4, 5), (193, 4, 5), (4, 4, 4), (2, 3, 62)])
def test_fields(device, n):
    print("[gpu-test] fields", n, flush=True)
    lat = np.diag([0.5 * m for m in n])
    lat[0, 1] = 0.3
    s = systems.make_system(n, np.diag(np.diag(lat)), np.zeros((0, 3)), with_projectors=False)
    s.lattice = lat
    ham = inq_amd.ks_hamiltonian(s, max_bands=1)
    osys = O.System(s.n, s.lattice, s.vloc, s.tables)
    rho = density(n)
    d = torch.from_numpy(rho).to(device)
    assert close(tddft.poisson(ham, d).cpu().numpy(), osys.poisson(rho))
    for kind in ("pbe_x", "pbe_c", "pbe"):
        vxc, exc, nvxc = tddft.xc(ham, d, kind)
        rv, re = osys.xc(rho, kind)
        assert close(vxc.cpu().numpy(), rv), kind
        assert exc == pytest.approx(re, rel=TOL)
        assert nvxc == pytest.approx((rho * rv).sum() * s.volume / s.npoints, rel=TOL)
    vion = np.random.default_rng(2).standard_normal(n)
    psi = torch.ones(n + (1,), dtype=torch.complex128, device=device)
    for hartree in (True, False):
        for xc in (False, "lda", "pbe"):
            en = tddft.ks_potential(ham, torch.from_numpy(vion).to(device), d, hartree, xc)
            vks, ren = osys.ks_potential(vion, rho, hartree, xc)
            for key in ren:
                assert en[key] == pytest.approx(ren[key], rel=TOL, abs=TOL), (key, hartree, xc)
            # H of a constant is V: the potential that the handle holds
            assert close(ham(psi).cpu().numpy()[..., 0].real, vks)
    ham.close()
