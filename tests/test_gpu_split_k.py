"""Long contractions into few tiles, whose K slices the workspace bounds: the
propagation intermediates (v0 over all gammas and orbitals, the mean field over
N^2) and the adjoint of the fields, against the oracle: 1e-10 of the largest
value, the repository's FP64 parity; the adjoint through a job whose workspace
allows few slices against one whose workspace allows many."""
import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu


def _job(sysm, n, o, g, cap, terms=4, dt=0.01):
    job = E.EngineJob(n, (o, o), g, cap, "restricted", "rhf", terms, dt, "fp64")
    job.set_hamiltonian(0.0, sysm.h1, sysm.chol)
    job.set_trial(sysm.mo_up, None, sysm.rdm1())
    job.build_measurement()
    job.build_propagation()
    return job


@pytest.mark.parametrize("n,o,g,cap", [(9, 2, 1, 1), (37, 5, 40, 1), (65, 7, 33, 300), (130, 11, 90, 4)])
def test_propagation_intermediates(n, o, g, cap):
    print(f"[split-k] {n} {o} {g} {cap}", flush=True)
    sysm = syn.make_system(n, o, g, seed=n)
    job = _job(sysm, n, o, g, cap)
    ref = O.propagation_intermediates(0.0, sysm.h1, sysm.chol, sysm.rdm1(), 0.01)
    got = job.get(5, 0).cpu().numpy().reshape(n, n)
    assert np.max(np.abs(got - ref["exp_h1"])) < 1e-10 * np.max(np.abs(ref["exp_h1"]))


@pytest.mark.parametrize("n,o,g,w", [(33, 4, 17, 3), (70, 9, 70, 5)])
def test_adjoint_of_fields(n, o, g, w):
    print(f"[split-k] adjoint {n} {o} {g} {w}", flush=True)
    sysm = syn.make_system(n, o, g, seed=n)
    up = torch.as_tensor(syn.perturbed_walkers(sysm.mo_up, w, 0.05, 1)).cuda()
    weights = torch.ones(w, dtype=torch.float64, device="cuda")
    fields = torch.as_tensor(np.random.default_rng(n).standard_normal((1, 2, w, g))).cuda()
    out = []
    for cap in (w, 64 * w):
        job = _job(sysm, n, o, g, cap)
        job.set_batch(w)
        f, gh1, gl = job.segment_energy_vjp(up, weights, -1.0, fields, want_grad=True)
        out.append((f.cpu(), gh1.cpu(), gl.cpu()))
        job.close()
    for a, b in zip(*out):
        assert (a - b).abs().max() <= 1e-11 * b.abs().max()
