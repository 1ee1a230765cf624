"""Runs near the memory of the device: arrays that only save time give way.

A handle whose orbital arrays take a good part of the memory keeps three of them
(its propagation then keeps two powers of a Taylor chain instead of three, with
the same bits).
"""
import numpy as np
import pytest
import torch

import inq_amd
from inq_amd import operations, systems

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
