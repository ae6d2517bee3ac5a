"""Boundary MPS at the block sizes where the truncation's eigensolver changes
form: sectors of up to 16 (one wave for both), up to 32 (a wave each), above
(D = 3, chi > 16), sectors of unequal size (D = 3), odd sizes and fewer
singular values than chi (right edge).

Tolerance: as for every truncated amplitude, ln|psi| within 1e-8 of the
oracle's QR / SVD boundary MPS where all its singular-value gaps are at least
1e-6."""
import numpy as np
import pytest
import torch

from helpers import random_configs
from test_bmps_gpu import _check, _oracle, _plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Lx,Ly,D,chi", [
    (6, 4, 2, 2), (8, 8, 2, 12), (5, 4, 4, 4), (4, 6, 4, 7), (5, 4, 3, 8), (6, 6, 3, 10),
    (5, 4, 4, 12), (7, 6, 3, 13), (7, 6, 3, 21),
    # fewer singular values than chi: nothing is lost
    (6, 4, 2, 6), (10, 4, 2, 16), (10, 4, 2, 20)])
def test_bmps_block_sizes(device, Lx, Ly, D, chi):
    m, sh, th = _plain(Lx, Ly, D, chi, 7 + Lx + 10 * D + chi, device)
    x = random_configs(np.random.default_rng(11), 20, sh.N, sh.N // 2, sh.N // 2)
    s, l = m.forward_log(torch.tensor(x, device=device))
    so, lo, go = _oracle(sh, th, x, chi)
    _check(s, l, so, lo, go)
