"""Options of an fPEPS or NN-fTNS changed on a live model (eta, activation, bmps_cache) take
effect at the next call, with the parameters where they were.  Tolerance: ln|psi| as in the
amplitude tests, 1e-9; the factored log-derivative against the dense one, 1e-10."""
import numpy as np
import pytest
import torch

from helpers import random_configs
from oracle import fpeps as fp
from test_fpeps_gpu import _nn
from vmc_torch_amd import fPEPS_Model_GPU

pytestmark = pytest.mark.gpu


def test_nnftns_options_take_effect(device):
    Lx, Ly, D, H = 3, 3, 2, 16
    m, sh, th, nn = _nn(Lx, Ly, D, H, 3, device, eta=0.5)
    x = random_configs(np.random.default_rng(2), 20, 9, 4, 4)
    xd = torch.tensor(x, device=device)
    for eta, act in ((0.5, "relu"), (0.9, "relu"), (0.9, "tanh"), (0.2, "tanh")):
        m.nn_eta, m.act_name = eta, act
        s, l = m.forward_log(xd)
        want = np.array([fp.nnftn_amplitude(sh, th, nn, eta, c, act) for c in x])
        assert np.array_equal(s.cpu().numpy(), np.sign(want))
        assert np.abs(l.cpu().numpy() - np.log(np.abs(want))).max() < 1e-9
        st = m.walker_state(xd)
        assert torch.equal(st["logabs"], l)
        O, _ = m.log_derivative(xd)
        F, _ = m.log_derivative_factored(xd)
        assert float((F.materialize() - O).norm() / O.norm()) < 1e-10


def test_bmps_cache_option_takes_effect(device):
    m = fPEPS_Model_GPU(6, 4, 2, generator=torch.Generator().manual_seed(1), max_bond=2).to(device)
    x = torch.tensor(random_configs(np.random.default_rng(2), 50, 24, 12, 12), device=device)
    m.forward_log(x)
    assert m._struct_obj.bmps_nocache == 0
    m.bmps_cache = False
    m.forward_log(x)
    assert m._struct_obj.bmps_nocache == 1
