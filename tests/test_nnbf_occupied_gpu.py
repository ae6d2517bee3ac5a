"""FP64 layers of the NNBF network on the matrix cores, with the outputs of
the occupied orbitals alone (libvmcx through vmc_torch_amd.NNBF_GPU), against
the FP64 oracle.

The sum over the hidden units is taken in another order than the oracle's:
ln|psi| then differs by at most n_f cond(A) H eps, 1e-10 for the matrices
here (cond < 1e4, H n_f <= 2^14), and signs are the same.
"""
import numpy as np
import pytest
import torch

from helpers import random_configs
from oracle import nnbf as onn
from vmc_torch_amd import NNBF_GPU

pytestmark = pytest.mark.gpu


# one, two, three and four column tiles, with one output, full tiles and one more than
# full; one k-step, a part of a chunk of the sum, several chunks
@pytest.mark.parametrize("Lx,Ly,nu,nd,hidden,act", [
    (4, 4, 1, 0, 16, "tanh"), (4, 4, 9, 7, 48, "relu"), (6, 5, 9, 8, 80, "tanh"),
    (6, 6, 16, 16, 256, "relu"), (8, 6, 17, 16, 64, "relu"), (8, 6, 24, 24, 16, "tanh"),
    (9, 6, 25, 24, 32, "relu"), (8, 8, 40, 24, 144, "relu")])
def test_occupied_outputs(device, Lx, Ly, nu, nd, hidden, act):
    g = torch.Generator().manual_seed(7)
    m = NNBF_GPU(Lx * Ly, nu + nd, hidden_dim=hidden, activation=act, bf_scale=0.3, gemm="fp64",
                 init="xavier", m_std=0.3, generator=g, chunk=1 << 15)
    with torch.no_grad():
        for p in m.params:
            if p.dim() == 1:
                p.copy_(0.05 * torch.randn(p.shape, generator=g, dtype=p.dtype))
    m = m.to(device)
    params = [p.detach().double().cpu().numpy() for p in m.params]
    rng = np.random.default_rng(3)
    x = random_configs(rng, 48, Lx * Ly, nu, nd)
    so, lo, _ = onn.forward(params, x, 2, m.bf_scale, act)
    # edges of tiles, of the blocks of rows (128, 256, 1024) and of the three size classes
    for rows in (1, 15, 17, 129, 1024, 1025, 2049, 16384, 16385, 17409):
        pick = rng.integers(0, len(x), rows)
        s, l = m.forward_log(torch.tensor(x[pick], device=device))
        assert np.array_equal(s.cpu().numpy(), so[pick]), rows
        assert np.abs(l.cpu().numpy() - lo[pick]).max() < 1e-10, rows


def test_occupied_outputs_wrong_count(device):
    """A row with too many or too few electrons is reported and leaves the others alone."""
    g = torch.Generator().manual_seed(5)
    m = NNBF_GPU(36, 32, hidden_dim=32, bf_scale=0.3, gemm="fp64", init="xavier", m_std=0.3,
                 generator=g).to(device)
    x = random_configs(np.random.default_rng(1), 40, 36, 16, 16)
    good = m.forward_log(torch.tensor(x, device=device))
    bad = x.copy()
    bad[3] = 3
    bad[17] = 0
    s, l = m.forward_log(torch.tensor(bad, device=device))
    keep = [r for r in range(40) if r not in (3, 17)]
    assert torch.isnan(l[[3, 17]]).all()
    assert torch.equal(s[keep], good[0][keep]) and torch.equal(l[keep], good[1][keep])


# the 64-lane elimination: one column in the last panel, full panels, one more
@pytest.mark.parametrize("nu,nd", [(17, 16), (24, 24), (25, 24), (32, 32)])
def test_determinant_panels(device, nu, nd):
    """Entries that leave no choice of pivot (one nonzero per row and column, in random
    order), so that sign and magnitude are exact up to the logarithms' rounding, 1e-12 of a
    sum of at most 64; the same with an empty column is singular."""
    rng = np.random.default_rng(nu)
    nf, N = nu + nd, 64
    x = np.zeros((6, N), np.int64)
    M = np.zeros((2 * N, nf))
    sites_up, sites_dn = rng.permutation(N)[:nu], rng.permutation(N)[:nd]
    x[:, sites_up] += 2
    x[:, sites_dn] += 1
    orb = np.concatenate([np.sort(sites_up), N + np.sort(sites_dn)])
    perm = rng.permutation(nf)
    M[orb, perm] = rng.choice([-1.0, 1.0], nf) * np.exp2(rng.integers(-3, 4, nf))
    A = M[orb]
    for empty in (None, 0, nf - 1):
        Me = M.copy()
        if empty is not None:
            Me[:, empty] = 0
        for gemm in ("fp64", "bf16"):
            m = NNBF_GPU(N, nf, hidden_dim=32, bf_scale=0.0, gemm=gemm, init="xavier").to(device)
            with torch.no_grad():
                [p for p in m.params if tuple(p.shape) == Me.shape][0].copy_(torch.tensor(Me))
            s, l = m.forward_log(torch.tensor(x, device=device))
            if empty is None:
                so, lo = np.linalg.slogdet(A)
                assert (s.cpu().numpy() == so).all()
                assert np.abs(l.cpu().numpy() - lo).max() < 1e-12 * max(1.0, 64 * np.log(8.0))
            else:
                assert (s == 0).all() and (l.cpu().numpy() == np.log(1e-45)).all()
