"""FP32 Slater determinants with M in another memory order (the FP64 copy that the kernels
read is contiguous): amplitudes, walker state and log-derivative bit for bit those of the
contiguous M, also after a change of its values."""
import numpy as np
import pytest
import torch

from helpers import random_configs
from vmc_torch_amd import SlaterDeterminant_GPU

pytestmark = pytest.mark.gpu


def test_fp32_m_of_another_order(device):
    N, nu, nd = 16, 7, 7
    x = torch.tensor(random_configs(np.random.default_rng(1), 50, N, nu, nd), device=device)
    a = SlaterDeterminant_GPU(2 * N, nu + nd, dtype=torch.float32).to(device)
    b = SlaterDeterminant_GPU(2 * N, nu + nd, dtype=torch.float32).to(device)
    b.params[0].data = a.params[0].data.t().contiguous().t()
    assert not b.params[0].is_contiguous()
    for _ in range(2):
        assert torch.equal(a.forward_log(x)[1], b.forward_log(x)[1])
        assert torch.equal(a.walker_state(x).logabs, b.walker_state(x).logabs)
        assert torch.equal(a.log_derivative(x)[0], b.log_derivative(x)[0])
        with torch.no_grad():
            a.params[0] *= 1.25
            b.params[0] *= 1.25
