"""The learned proposal on fPEPS and NN-fTNS models: one injected step against the oracle's
Metropolis-Hastings step with the oracle's amplitudes (configurations and acceptances
identical, the uniforms 1e-4 away from every boundary), then free-running steps of one and two
moves, whose amplitudes are those of the walkers that they end at (1e-9 in ln|psi|)."""
import numpy as np
import pytest
import torch

from helpers import random_configs
from oracle import fpeps as fp
from oracle import proposal as op
from test_fpeps_gpu import _nn, _plain
from test_proposal_gpu import _net
from vmc_torch_amd import fPEPS_Model_GPU, fPEPS_Model_reuse_GPU
from vmc_torch_amd.sampler import LearnedProposalSamplerGPU

pytestmark = pytest.mark.gpu


def _model(kind, device):
    if kind == "nnftns":
        m, sh, th, nn = _nn(3, 3, 2, 16, 5, device)

        def amps(x):
            a = np.array([fp.nnftn_amplitude(sh, th, nn, m.nn_eta, c) for c in x])
            return np.sign(a), np.log(np.abs(a))
        return m, 3, 3, amps
    if kind == "bmps":
        sh = fp.PEPSShape(4, 3, 2)
        th = fp.random_theta(sh, np.random.default_rng(5))
        m = fPEPS_Model_GPU(4, 3, 2, theta=th, max_bond=2).to(device)
        assert m._bmps
        return m, 4, 3, lambda x: fp.bmps_log_amplitudes(sh, th, x, 2)[:2]
    m, sh, th = _plain(3, 4, 2, 5, device)
    if kind == "reuse":
        m = fPEPS_Model_reuse_GPU(3, 4, 2, theta=th).to(device)

    def amps(x):
        a = fp.amplitudes(sh, th, np.asarray(x))
        return np.sign(a), np.log(np.abs(a))
    return m, 3, 4, amps


@pytest.mark.parametrize("kind", ["fpeps", "reuse", "bmps", "nnftns"])
def test_learned_steps(device, kind):
    model, Lx, Ly, amps = _model(kind, device)
    N, C, B = Lx * Ly, 8, 24
    th, P = _net(C, 5, scale=2.0)
    th32 = P.double().numpy()
    rng = np.random.default_rng(7)
    x0 = random_configs(rng, B, N, N // 3, N // 3)

    def logamp(c):
        return amps(np.asarray(c)[None])[1][0]
    uc, ua = rng.random(B), rng.random(B)
    want = []
    for b in range(B):
        lf, vf, _ = op.forward(th32, C, Lx, Ly, x0[b])
        cdf = np.cumsum(np.exp(op.log_q(lf, vf))[vf])
        while np.min(np.abs(cdf - uc[b])) < 1e-4:
            uc[b] = rng.random()
        mv = op.sample_move(op.log_q(lf, vf), uc[b])
        xp = op.apply_move(x0[b], Lx, Ly, mv)
        lr, vr, _ = op.forward(th32, C, Lx, Ly, xp)
        r = np.exp(2 * (logamp(xp) - logamp(x0[b])) + op.log_q(lr, vr)[mv] - op.log_q(lf, vf)[mv])
        if abs(ua[b] - r) < 1e-4 * max(r, 1e-300):
            ua[b] = 0.5 * min(r, 1.0)
        want.append(op.mh_step(th32, C, Lx, Ly, x0[b], logamp, uc[b], ua[b]))
    xd = torch.tensor(x0, device=device)
    s = LearnedProposalSamplerGPU(Lx, Ly, channels=C, params=P.to(device))
    s.sweeps(xd, model, 1, draws=[(torch.tensor(uc, device=device),
                                   torch.tensor(ua, device=device))])
    assert np.array_equal(xd.cpu().numpy(), np.array([w[0] for w in want]))
    assert np.array_equal(s.last_acceptance[0].cpu().numpy(), np.array([w[1] for w in want]))
    for moves in (1, 2):
        s = LearnedProposalSamplerGPU(Lx, Ly, channels=C, params=P.to(device), seed=3,
                                      moves_per_proposal=moves)
        sign, logabs = s.sweeps(xd, model, 5)
        so, lo = amps(xd.cpu().numpy())
        assert np.array_equal(sign.cpu().numpy(), so)
        assert np.abs(logabs.cpu().numpy() - lo).max() < 1e-9
