"""v0 = 1/2 sum_g L_g L_g in chunks of what the VHS buffer holds (two Cholesky
indices a walker): one chunk, several with a short last one, the most that are
taken (eight), and few walkers, for which a buffer of its own is allocated.
exp(-dt/2 h1_mod) with dt = 2, so that v0 enters it undamped, against the oracle
(1e-10 of the largest value, the repository's FP64 parity)."""
import numpy as np
import pytest

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,g,w", [(12, 40, 20), (12, 41, 20), (12, 48, 3), (12, 49, 3), (33, 33, 16), (33, 100, 7)])
def test_propagation_intermediates(n, g, w):
    print(f"[v0] {n} {g} {w}", flush=True)
    s = syn.make_system(n, 4, g, seed=n + g)
    job = E.EngineJob(n, (4, 4), g, w, "restricted", "rhf", 6, 2.0, "fp64")
    job.set_hamiltonian(0.0, s.h1, s.chol)
    job.set_trial(s.mo_up, None, s.rdm1())
    job.build_measurement()
    job.build_propagation()
    ref = O.propagation_intermediates(0.0, s.h1, s.chol, s.rdm1(), 2.0)["exp_h1"]
    got = job.get(5, 0).cpu().numpy().reshape(n, n)
    assert np.max(np.abs(got - ref)) < 1e-10 * np.max(np.abs(ref))
