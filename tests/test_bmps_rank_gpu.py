"""Boundary MPS on states whose truncation loses nothing: a D = 2 state written with D = 4 (every
bond through an isometry within its parity sectors) and chi = 8, the rank of three rows of
it.  Each eigensolve of the truncation meets a block of half its rank or less, the rest
rounding noise; the amplitudes are those of the D = 2 state with no truncation (chi = 16).

Tolerance: the rounding of a block's entries is at most about 16 ulp of its diagonal, so a
noise column of the factor has a square of at most (16 ulp)^2 / 1 ulp (a pivot exceeds one ulp
of its row's diagonal).  It can push out of the chi kept directions one of at most that
eigenvalue, 256 ulp, that is a part sqrt(256 * 2.2e-16) = 2.4e-7 of the boundary: 1e-6 for the
worst amplitude.  A pivot below the noise has no such bound: it moved one of these amplitudes
by 1.1e-5."""
import numpy as np
import pytest
import torch

from helpers import random_configs
from oracle import fpeps as fp
from vmc_torch_amd import fPEPS_Model_GPU

pytestmark = pytest.mark.gpu


def widened(Lx, Ly, rng):
    """theta of a random D = 2 state of nonnegative entries, and of the same state with D = 4."""
    s2, s4 = fp.PEPSShape(Lx, Ly, 2), fp.PEPSShape(Lx, Ly, 4)
    th2 = fp.random_theta(s2, rng)
    bond = {}

    def isometry(key):
        if key not in bond:
            a = rng.uniform(0.3, 1.2, 2)
            V = np.zeros((4, 2))
            V[:2, 0] = np.cos(a[0]), np.sin(a[0])
            V[2:, 1] = np.cos(a[1]), np.sin(a[1])
            bond[key] = V
        return bond[key]

    out = []
    for i, (m2, m4) in enumerate(zip(s2.masks, s4.masks)):
        x, y = divmod(i, Ly)
        t = np.zeros(m2.shape)
        t[m2] = np.abs(th2[s2.offsets[i]:s2.offsets[i + 1]])
        th2[s2.offsets[i]:s2.offsets[i + 1]] = t[m2]
        for ax, key in ((1, ("h", x, y)), (2, ("v", x, y)), (3, ("v", x + 1, y)),
                        (4, ("h", x, y + 1))):
            if t.shape[ax] == 2:
                t = np.moveaxis(np.tensordot(isometry(key), t, (1, ax)), 0, ax)
        assert t.shape == m4.shape and not t[~m4].any()
        out.append(t[m4])
    return th2, np.concatenate(out)


def test_noise_does_not_displace(device):
    worst = []
    for seed in (1, 2, 3, 4):
        a, b = widened(6, 6, np.random.default_rng(seed))
        x = torch.tensor(random_configs(np.random.default_rng(seed), 8192, 36, 18, 18), device=device)
        s0, l0 = fPEPS_Model_GPU(6, 6, 2, theta=a, max_bond=16).to(device).forward_log(x)
        s, l = fPEPS_Model_GPU(6, 6, 4, theta=b, max_bond=8).to(device).forward_log(x)
        worst.append(float((s * s0 * torch.exp(l - l0) - 1).abs().max()))
    assert max(worst) < 1e-6, worst
