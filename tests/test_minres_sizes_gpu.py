"""MINRES at the sizes where its launches change: strides of 256 columns, one to four
first-stage blocks of a dot (2048 columns each), four rows a workgroup and the last of them
alone, fewer rows than chunks, and rows beyond the short form's widest (Np > 8192).  A few
iterations against the oracle; the updates of whole solves are in test_minres_sums_gpu.py.

Tolerance: four iterations amplify the FP64 rounding of sums over Np terms by
the ratio of the Krylov vectors' scales, about 1e3 here: 1e3 * 2^-53 *
sqrt(Np) < 1e-11 relative; the bound is 1e-10."""
import numpy as np
import pytest
import torch

from oracle import sr as osr
from test_sr_gpu import _problem, _rel
from vmc_torch_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("Ns,Np", [
    (2, 1), (1, 1024), (127, 1025), (129, 2048), (257, 3071), (300, 3073), (513, 4097),
    (130, 6145), (384, 8192), (200, 8193), (1031, 17)])
def test_minres_sizes(device, Ns, Np, dtype):
    O, E = _problem(Ns, Np, 7 + Ns + Np)
    Od = torch.tensor(O, device=device).to(dtype)
    O = Od.cpu().double().numpy()
    iters = min(4, Ns - 1 if Ns > 1 else 1)
    want, winfo = osr.sr_minres(O, E, float(E.mean()) + 0.25, 1e-2, rtol=1e-14, maxiter=iters)
    dp, stats, info = kernels.sr_minres(Od, torch.tensor(E, device=device),
                                        float(E.mean()) + 0.25, 1e-2, rtol=1e-14, maxiter=iters)
    assert int(info.item()) == winfo
    assert _rel(dp.cpu().numpy(), want) < 1e-10
