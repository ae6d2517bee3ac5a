"""Exact fPEPS in FP64 from the column table, parameters scaled by a power of two s: psi is
of degree one in every site's tensor, so ln|psi| grows by N ln s, the signs and the local
energies stay, and below the smallest amplitude (1e-45) ln|psi| is its logarithm and the sign
is still psi's.  s = 2^140 takes the product of eight slices out of FP64's range, that of four
(one column of the network) does not.

Tolerance: ln|psi| to 4 ulp of its largest part, N ln s < 3200, 2e-12; local energies are
ratios of the same amplitudes, 1e-9."""
import numpy as np
import pytest
import torch

from helpers import random_configs
from vmc_torch_amd import fPEPS_Model_GPU
from vmc_torch_amd.hamiltonian import spinful_Fermi_Hubbard_square_lattice_torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Lx,Ly,D", [(2, 1, 2), (2, 2, 4), (3, 4, 2), (4, 3, 2), (4, 4, 4), (4, 6, 3),
                                     (4, 8, 2)])
def test_scaled_parameters(device, Lx, Ly, D):
    N = Lx * Ly
    nu, nd = (N + 1) // 2, N // 2
    m = fPEPS_Model_GPU(Lx, Ly, D, generator=torch.Generator().manual_seed(5)).to(device)
    x = torch.tensor(random_configs(np.random.default_rng(1), 60, N, nu, nd), device=device)
    H = spinful_Fermi_Hubbard_square_lattice_torch(Lx, Ly, 1.0, 8.0, nu + nd,
                                                   n_fermions_per_spin=(nu, nd))
    H.precompute_hops_gpu(device)
    p = m.params[0]
    with torch.no_grad():
        p *= 4.0
    s0, l0 = m.forward_log(x)
    e0 = m.local_energy(x, H)
    assert float(l0.min()) > np.log(1e-44)
    with torch.no_grad():
        p *= 2.0 ** 140
    s1, l1 = m.forward_log(x)
    e1 = m.local_energy(x, H)
    assert torch.equal(s0, s1)
    assert float((l1 - l0 - N * 140 * np.log(2.0)).abs().max()) < 2e-12
    assert float(((e1 - e0) / (1 + e0.abs())).abs().max()) < 1e-9
    with torch.no_grad():
        p *= 2.0 ** -280
    s2, l2 = m.forward_log(x)
    assert torch.equal(s0, s2)
    assert bool((l2 == np.log(1e-45)).all())
