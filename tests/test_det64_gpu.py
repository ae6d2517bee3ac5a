"""FP64 determinants of 33 to 64 electrons: eliminated in panels, each entry takes the
multiply-adds of the unblocked elimination, in its order.  Nearly singular matrices (one
column of M within 1e-9 of the span of the others) show it: another order moves ln|psi| by
1e-7 to 1e-5.

Oracle: the unblocked elimination with the device's choice of pivots, fused multiply-adds
formed exactly.  Tolerance: the pivots being the same bits, what remains is the rounding of 64
logarithms of at most 25 and of their sum, 64 * 25 * 2^-52 < 4e-13; the bound is 1e-12."""
import numpy as np
import pytest
import torch

from helpers import random_configs
from vmc_torch_amd import NNBF_GPU, kernels


def _two_sum(a, b):
    s = a + b
    t = s - a
    return s, (a - (s - t)) + (b - t)


def fma(a, b, c):
    """Correctly rounded a b + c of doubles far from overflow and underflow (Boldo and
    Melquiond, IEEE Trans. Comput. 57, 2008: exact product and sums, the small part rounded
    to odd)."""
    def split(v):
        w = v * 134217729.0
        h = w - (w - v)
        return h, v - h
    p = a * b
    (ah, al), (bh, bl) = split(a), split(b)
    e = ((ah * bh - p) + ah * bl + al * bh) + al * bl
    th, tl = _two_sum(c, e)
    vh, vl = _two_sum(p, th)
    z, r = _two_sum(tl, vl)
    even = (np.ascontiguousarray(z).view(np.int64) & 1) == 0
    z = np.where((r != 0) & even, np.nextafter(z, np.where(r > 0, np.inf, -np.inf)), z)
    return vh + z


def unblocked(A):
    """Pivots of the elimination of A[b][lane][step] ([B][64][64])."""
    A = A.copy()
    B = len(A)
    lane = np.arange(64, dtype=np.uint32)
    b = np.arange(B)
    piv = np.zeros((B, 64))
    for p in range(64):
        key = (np.abs(A[:, :, p]).astype(np.float32).view(np.uint32) & ~np.uint32(63)) | (63 - lane)
        q = 63 - (key.max(1) & 63).astype(int)
        row = A[b, q].copy()
        piv[b, q] = row[:, p]
        f = A[:, :, p] / row[:, p, None]
        f[b, q] = 1.0
        A[:, :, p + 1:] = fma(-f[:, :, None], row[:, None, p + 1:], A[:, :, p + 1:])
    return piv


def test_fma_is_exact():
    from fractions import Fraction
    r = np.random.RandomState(3)
    a, b = r.standard_normal(400), r.standard_normal(400)
    c = -a * b * (1 + r.randint(-2, 3, 400) * 2.0 ** -r.randint(1, 60, 400))
    for x, y, z, w in zip(a, b, c, fma(a, b, c)):
        assert float(Fraction(x) * Fraction(y) + Fraction(z)) == w


@pytest.mark.gpu
@pytest.mark.parametrize("N,nu,nd", [(49, 17, 16), (64, 25, 25), (64, 32, 32)])
def test_panels_keep_the_order(device, N, nu, nd):
    nf = nu + nd
    r = np.random.RandomState(nf)
    M = r.standard_normal((2 * N, nf))
    M[:, -1] = M[:, :-1] @ r.standard_normal(nf - 1) + 1e-9 * r.standard_normal(2 * N)
    x = random_configs(np.random.default_rng(5), 24, N, nu, nd)
    A = np.tile(np.eye(64), (len(x), 1, 1))
    for k, c in enumerate(x):
        orb = np.concatenate([np.flatnonzero(c & 2), N + np.flatnonzero(c & 1)])
        A[k, :nf, :nf] = M[orb].T
        A[k, :nf, nf:] = A[k, nf:, :nf] = 0.0
    want = np.log(np.abs(unblocked(A))).sum(1)
    xd, Md = torch.tensor(x, device=device), torch.tensor(M, device=device)
    _, got = kernels.slater_refresh(Md, xd)
    assert np.abs(got.cpu().numpy() - want).max() < 1e-12
    m = NNBF_GPU(N, nf, hidden_dim=16, bf_scale=0.0, gemm="fp64", init="xavier").to(device)
    with torch.no_grad():
        next(p for p in m.params if tuple(p.shape) == M.shape).copy_(Md)
    _, got = m.forward_log(xd)
    assert np.abs(got.cpu().numpy() - want).max() < 1e-12
