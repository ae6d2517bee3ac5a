"""The device-side checks that replace host comparisons: parameters against
the copy a walker state was built from, and non-finite samples.  Exact
(counts, bit comparisons; a rebuilt state equals a fresh model's bit for
bit)."""
import pytest
import torch

from vmc_torch_amd import (MetropolisExchangeSpinfulSamplerGPU, SlaterDeterminant_GPU,
                           evaluate_energy, fPEPS_Model_GPU, kernels)
from vmc_torch_amd.hamiltonian import spinful_Fermi_Hubbard_square_lattice_torch
from vmc_torch_amd.vmc_utils import check_grads_amps, initialize_walkers, random_initial_config

pytestmark = pytest.mark.gpu


def _setup(device, make, B=40):
    H = spinful_Fermi_Hubbard_square_lattice_torch(4, 3, 1.0, 8.0, 12, n_fermions_per_spin=(6, 6))
    fxs = initialize_walkers(lambda seed: random_initial_config(12, 12, seed=seed), B, seed=3,
                             device=device)
    return H, fxs, make().to(device)


MODELS = {
    "slater64": lambda: SlaterDeterminant_GPU(24, 12, generator=torch.Generator().manual_seed(1)),
    "slater32": lambda: SlaterDeterminant_GPU(24, 12, dtype=torch.float32,
                                              generator=torch.Generator().manual_seed(1)),
    "fpeps": lambda: fPEPS_Model_GPU(4, 3, 2, generator=torch.Generator().manual_seed(1)),
    "fpeps32": lambda: fPEPS_Model_GPU(4, 3, 2, generator=torch.Generator().manual_seed(1),
                                       amp="fp32"),
}


@pytest.mark.parametrize("write", ["data", "single", "optimizer"])
@pytest.mark.parametrize("name", list(MODELS))
def test_parameter_changes_are_seen(device, name, write):
    H, fxs, m = _setup(device, MODELS[name])
    smp = MetropolisExchangeSpinfulSamplerGPU(seed=5)
    smp.step(fxs, m, H.graph)
    m.forward_log(fxs)
    m.log_derivative(fxs)
    p = m.params[0]
    if write == "data":
        p.data.mul_(1.25)
        p.data.view(-1)[3] += 0.5
    elif write == "single":
        p.data.view(-1)[p.numel() - 1] *= -1.0
    else:
        with torch.no_grad():
            p.sub_(0.1 * torch.randn(p.shape, generator=torch.Generator().manual_seed(2),
                                     dtype=p.dtype).to(device))
    m.forward_log(fxs)          # must not hide the change from the walker state
    fresh = MODELS[name]().to(device)
    fresh.params[0].data.copy_(p.data)
    E, want = evaluate_energy(fxs, m, H)[1], evaluate_energy(fxs, fresh, H)[1]
    assert torch.equal(E, want)
    O, (s, l) = m.log_derivative(fxs)
    Of, (sf, lf) = fresh.log_derivative(fxs)
    assert torch.equal(O, Of) and torch.equal(s, sf) and torch.equal(l, lf)
    n0 = m.accept_counts(fxs).clone()
    a = smp.step(fxs.clone(), m, H.graph, use_log_amp=True)
    smp.sweep_counter -= 1
    b = smp.step(fxs.clone(), fresh, H.graph, use_log_amp=True)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1][1], b[1][1])
    assert (m._state["n_accept"] if name.startswith("f") else m._state.n_accept).ge(n0).all()


@pytest.mark.parametrize("name", ["slater64", "slater32"])
def test_unchanged_parameters_keep_the_state(device, name):
    """A sweep's incremental state is not rebuilt while M stands."""
    H, fxs, m = _setup(device, MODELS[name])
    smp = MetropolisExchangeSpinfulSamplerGPU(seed=5, refresh_every=0)
    smp.step(fxs, m, H.graph)
    ainv = m._state.ainv.clone()
    evaluate_energy(fxs, m, H)
    m.log_derivative(fxs)
    m.forward_log(fxs)
    assert torch.equal(ainv, m._state.ainv)
    assert int(m._state.since_refresh.max()) < kernels.SLATER_STALE
    m.invalidate()
    m.walker_state(fxs)
    assert int(m._state.since_refresh.max()) == 0


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("B,n,ld", [(1, 1, 1), (5, 0, 3), (7, 129, 129), (66, 64, 80), (9, 33, 35)])
def test_count_nonfinite(device, dtype, B, n, ld):
    g = torch.Generator().manual_seed(B + n)
    wide = torch.randn(B, ld, generator=g).to(dtype)
    O = wide.to(device)[:, :n]
    s, l = torch.ones(B, dtype=torch.float64, device=device), torch.zeros(B, dtype=torch.float64,
                                                                          device=device)
    assert kernels.count_nonfinite(O, s, l).tolist() == [0, 0]
    check_grads_amps(O, s, l)
    bad = 0
    for k, v in enumerate((float("nan"), float("inf"), -float("inf"))):
        if n and k < B:
            O[k, (n - 1) * k // 2] = v
            bad += 1
    s[B - 1] = float("nan")
    assert kernels.count_nonfinite(O, s, l).tolist() == [1, bad]
    with pytest.raises(ValueError, match="amplitudes"):
        check_grads_amps(O, s, l, torch.zeros(B, 2))
    if bad:
        with pytest.raises(ValueError, match=f"{bad}/{B} samples"):
            check_grads_amps(O, torch.ones_like(s), l)
