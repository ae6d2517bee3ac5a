"""Exact FP64 fPEPS amplitudes and sweeps from the column table (one wave per
configuration) over every shape of a half: one or two rows, D = 1 .. 4 (D = 3:
unequal parities), one to eight columns, more edges than one launch takes.

Tolerances: FP64 both sides, amplitudes |ln psi| within 1e-10 of the oracle
(sums of at most D^8 terms in another order; configurations whose amplitude is
below 1e-8 of the largest are sums with cancellation and are left out);
sweeps on tie-free draws: the oracle's configurations and signs exactly."""
import numpy as np
import pytest
import torch

from helpers import random_configs, tie_free_draws
from oracle import fpeps as fp
from oracle import hubbard as ohub
from oracle import sampler as osamp
from vmc_torch_amd import fPEPS_Model_GPU

pytestmark = pytest.mark.gpu


def _case(Lx, Ly, D, seed, device, scale=1.0):
    sh = fp.PEPSShape(Lx, Ly, D)
    th = fp.random_theta(sh, np.random.default_rng(seed)) * scale
    return fPEPS_Model_GPU(Lx, Ly, D, theta=th).to(device), sh, th


@pytest.mark.parametrize("Lx,Ly,D,scale", [
    (2, 1, 2, 1.0), (2, 2, 1, 1.0), (2, 5, 3, 1.0), (2, 8, 4, 1.0), (3, 1, 4, 1.0),
    (3, 2, 3, 1.0), (3, 3, 2, 1.0), (3, 4, 4, 1.0), (4, 1, 3, 1.0), (4, 2, 4, 1.0),
    (4, 3, 3, 1.0), (4, 5, 2, 1.0), (4, 4, 4, 1e30), (4, 4, 3, 1e-18), (4, 8, 2, 1.0)])
def test_amplitudes(device, Lx, Ly, D, scale):
    m, sh, th = _case(Lx, Ly, D, 3 + Lx + 7 * Ly + D, device, scale)
    N = Lx * Ly
    n = N // 2 if N % 2 == 0 else N // 2 + (N // 2) % 2
    x = random_configs(np.random.default_rng(5), 33, N, n, n) if D > 1 else \
        3 * (np.random.default_rng(5).random((33, N)) < 0.5).astype(np.int64)
    s, l = m.forward_log(torch.tensor(x, device=device))
    s, l = s.cpu().numpy(), l.cpu().numpy()
    # in units of `scale` per tensor, so that the oracle does not overflow
    want = fp.amplitudes(sh, th / scale, x)
    lo = np.log(1e-45)
    for a, si, li in zip(want, s, l):
        if a == 0.0 or abs(a) < 1e-8 * np.abs(want).max():
            continue
        lw = np.log(abs(a)) + N * np.log(scale)
        assert si == np.sign(a)
        assert abs(li - max(lw, lo)) < 1e-10 * max(1.0, abs(lw))


def test_vanishing_and_nonfinite(device):
    """An odd number of electrons, zero and infinite parameters: sign 0."""
    m, sh, th = _case(4, 3, 2, 1, device)
    x = torch.tensor(random_configs(np.random.default_rng(2), 9, 12, 6, 5), device=device)
    for value in (None, 0.0, float("inf"), float("nan")):
        if value is not None:
            with torch.no_grad():
                m.params[0].fill_(value)
        s, l = m.forward_log(x)
        assert torch.all(s == 0) and torch.all(l == np.log(1e-45))


@pytest.mark.parametrize("Lx,Ly,D,B,repeat", [(4, 4, 4, 37, 1), (3, 3, 3, 5, 1), (2, 4, 2, 9, 14)])
def test_sweep(device, Lx, Ly, D, B, repeat):
    m, sh, th = _case(Lx, Ly, D, 11, device)
    N = Lx * Ly
    n = (N // 2) & ~1
    x = random_configs(np.random.default_rng(8), B, N, n, n)
    edges = ohub.SquareLattice(Lx, Ly).sweep_edges() * repeat     # 140 edges in the last case

    def logamp(c):
        a = fp.amplitudes(sh, th, c)
        return np.sign(a), np.log(np.maximum(np.abs(a), 1e-45))
    draws, *_ = tie_free_draws(logamp, x, edges, 2, np.random.default_rng(9))
    want, ws, wl, wacc = osamp.sweep(logamp, x, edges, osamp.InjectedDraws(*draws), n_sweeps=2)
    f = torch.tensor(x, device=device)
    e = torch.tensor(edges, dtype=torch.int32, device=device)
    uc, bits, ua = draws
    d = (torch.tensor(uc, device=device), torch.tensor(bits, device=device),
         torch.tensor(ua, device=device))
    s, l, acc = m.mcmc_sweep(f, e, 2, 0, 0, draws=d)
    assert np.array_equal(f.cpu().numpy(), want)
    assert np.array_equal(s.cpu().numpy(), ws)
    assert np.abs(l.cpu().numpy() - wl).max() < 1e-9
    assert np.array_equal(acc.cpu().numpy(), wacc)
    # Philox: two sweeps in one call and one call each
    f1, f2 = torch.tensor(x, device=device), torch.tensor(x, device=device)
    l1 = m.mcmc_sweep(f1, e, 2, 77, 3)[1].clone()
    m.mcmc_sweep(f2, e, 1, 77, 3)
    l2 = m.mcmc_sweep(f2, e, 1, 77, 4)[1]
    px, ps, pl, _ = osamp.sweep(logamp, x, edges, osamp.PhiloxDraws(77, 3), n_sweeps=2)
    assert torch.equal(f1, f2) and torch.equal(l1, l2)
    assert np.array_equal(f1.cpu().numpy(), px)
