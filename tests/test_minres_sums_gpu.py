"""MINRES: one order of the sums at every size.  The update of a stiff problem is not
determined by its inputs (the Lanczos vectors lose their orthogonality over some tens of
iterations, so that another order of the sums moves it by per cents), hence the digests of
the updates and of the statistics, recorded from the form with one launch per operation, at
the sizes where the form changes: one and several 256-thread strides, one to four first-stage
blocks of a dot (2048 columns each), four rows a workgroup, the widest row of the short form
(8192) and beyond.

Tolerance: none, bit for bit (every operation is an IEEE one in a fixed order; the inputs
are quotients of integers, correctly rounded wherever they are formed)."""
import hashlib

import numpy as np
import pytest
import torch

from vmc_torch_amd import kernels

pytestmark = pytest.mark.gpu

DIGESTS = {
    (3, 1, "float64"): "54197a98fdd0377e", (3, 1, "float32"): "81cfe70f202730bd",
    (700, 255, "float64"): "4a635f3e61afd565", (700, 255, "float32"): "5610f302614933c5",
    (301, 256, "float64"): "54e258cea6a7ece7", (301, 256, "float32"): "34b6d3b18aa3f8c5",
    (514, 257, "float64"): "59378284c1a7a8b9", (514, 257, "float32"): "618be3e743844c9d",
    (1000, 2048, "float64"): "8bed2e53674f1d24", (1000, 2048, "float32"): "f8d54dffe95decf8",
    (999, 2049, "float64"): "a6202d8e40aefcd8", (999, 2049, "float32"): "c696f7ae41c57f3c",
    (700, 2160, "float64"): "c490743de982f395", (700, 2160, "float32"): "5387741cc2c6ff9d",
    (601, 4097, "float64"): "3fbcc77eea2d664b", (601, 4097, "float32"): "fc9af5f21b60f711",
    (402, 6145, "float64"): "104d543287f09607", (402, 6145, "float32"): "1f366de736b1e43e",
    (300, 8192, "float64"): "71bfd9ca5ad02968", (300, 8192, "float32"): "1e31633db36ca3a4",
    (301, 8193, "float64"): "fe10d268f1004ff0", (301, 8193, "float32"): "90848d1fb1b23039",
    (120, 40000, "float64"): "1d2a85de43e4b710", (120, 40000, "float32"): "8e0282c4ae2867b0",
}
SIZES = [(3, 1), (700, 255), (301, 256), (514, 257), (1000, 2048), (999, 2049), (700, 2160),
         (601, 4097), (402, 6145), (300, 8192), (301, 8193), (120, 40000)]


def problem(Ns, Np):
    """Heavy-tailed O and E (quotients of integers)."""
    r = np.random.RandomState(Ns + 10 * Np)
    O = r.randint(-1000, 1001, (Ns, Np)) / r.randint(1, 1001, (Ns, Np))
    O *= 1.0 / r.randint(1, 101, Np)
    E = r.randint(-1000, 1001, Ns) / r.randint(1, 101, Ns)
    return O, E


def solve(O, E, dtype, device, maxiter=100, rtol=1e-4):
    return kernels.sr_minres(torch.tensor(O, device=device).to(dtype),
                             torch.tensor(E, device=device), float(E.mean()), 1e-2, rtol=rtol,
                             maxiter=maxiter)


def digest(dp, stats):
    return hashlib.sha256(dp.cpu().numpy().tobytes() + stats.cpu().numpy().tobytes()).hexdigest()[:16]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("Ns,Np", SIZES)
def test_minres_recorded(device, Ns, Np, dtype):
    O, E = problem(Ns, Np)
    dp, stats, _ = solve(O, E, dtype, device)
    assert digest(dp, stats) == DIGESTS[Ns, Np, str(dtype)[6:]]


@pytest.mark.parametrize("Ns,Np", [(700, 2160), (301, 8193)])
def test_minres_stops_where_it_converges(device, Ns, Np):
    """Launches after convergence change nothing: a limit of as many iterations as were taken,
    one more, and many more give the same bits."""
    O, E = problem(Ns, Np)
    dp, stats, info = solve(O, E, torch.float64, device)
    it = int(stats[4])
    assert int(info) == 0 and it < 99
    for n in (it, it + 1, 400):
        dq, st, inf = solve(O, E, torch.float64, device, maxiter=n)
        assert int(inf) == 0
        assert torch.equal(dp, dq) and torch.equal(stats, st)
