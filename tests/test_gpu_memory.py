"""Runs near the memory of the device: arrays that only save time give way.

A handle whose orbital arrays take a good part of the memory keeps three of them
(its propagation then keeps two powers of a Taylor chain instead of three, with
the same bits), and an adjoint on a non-cubic grid whose tape fits only without the
transforms of the powers is created without them (1e-9 against the tape with them,
whose sums are formed in another order).
"""
import numpy as np
import pytest
import torch

import inq_amd
from inq_amd import adjoint, operations, systems

pytestmark = pytest.mark.gpu


def _system(n, projectors=True):
    lat = np.diag([0.4 * m for m in n])
    atoms = np.array([[1.0, 1.2, 0.8], [4.0, 3.0, 5.0]])
    return systems.make_system(n, lat, atoms, seed=7, with_projectors=projectors)


@pytest.mark.parametrize("n", [(48, 48, 48), (40, 36, 48)])
def test_few_orbital_arrays_where_memory_is_short(device, n):
    s = _system(n)
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    band = 16 * s.npoints
    many = int(free / 7.5) // band
    print("[gpu-test] memory", n, many, "bands,", free >> 30, "GiB free", flush=True)
    few = inq_amd.ks_hamiltonian(s, max_bands=8, tuning=None)
    before = torch.cuda.mem_get_info()[0]
    ham = inq_amd.ks_hamiltonian(s, max_bands=many, tuning=None)
    taken = before - torch.cuda.mem_get_info()[0]
    print("[gpu-test]   taken / orbital array %.2f" % (taken / (band * many)), flush=True)
    assert taken < 3.5 * band * many
    g = torch.Generator(device=device).manual_seed(3)
    psi = torch.randn(n + (8,), dtype=torch.complex128, device=device, generator=g)
    for order in (1, 2, 3, 4, 5, 7):
        a = operations.exponential_in_place(few, 0.01j, psi.clone(), order)
        b = operations.exponential_in_place(ham, 0.01j, psi.clone(), order)
        assert torch.equal(a, b), order
    ham.close()
    few.close()


def test_tape_without_transforms_where_memory_is_short(device):
    n, nst, order = (40, 36, 32), 16, 4
    s = _system(n)
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    step = 2 * order * 16 * s.npoints * nst  # tape of a step, powers alone
    steps = int(0.65 * free / step)
    print("[gpu-test] tape of", steps, "steps,", free >> 30, "GiB free", flush=True)
    psi = torch.from_numpy(systems.random_orbitals(s, nst, ecut=10.0, seed=2)).to(device)
    res = []
    for every in (steps, 20):
        ham = inq_amd.ks_hamiltonian(s, max_bands=nst, tuning=None)
        prop = adjoint.propagation_adjoint(ham, nst, nsteps=steps, dt=0.01, ncoef=3, omega=0.1,
                                           order=order, checkpoint_every=every)
        coef = torch.tensor([0.02, -0.01, 0.03], dtype=torch.float64, requires_grad=True)
        vloc = torch.from_numpy(s.vloc).to(device).requires_grad_(True)
        loss = adjoint.td_current_loss(coef, vloc, prop, psi)
        loss.backward()
        res.append((loss.item(), coef.grad.numpy().copy(), vloc.grad.cpu().numpy()))
        prop.close()
        ham.close()
        torch.cuda.empty_cache()
    (la, ca, va), (lb, cb, vb) = res
    assert abs(la - lb) <= 1e-9 * abs(lb)
    assert np.linalg.norm(ca - cb) <= 1e-9 * np.linalg.norm(cb)
    assert np.linalg.norm(va - vb) <= 1e-9 * np.linalg.norm(vb)
