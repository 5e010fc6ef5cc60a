"""Weights of a small FP64 job's step follow from the population-control shift
that it starts with; e_estimate enters only the shift that it leaves
(propagation.py:306-334).  So an e_estimate far from the shift, or not finite,
leaves the weights as they are: against the oracle, 1e-10 of the largest value,
the repository's FP64 parity."""
import math

import numpy as np
import pytest

from ad_afqmc_amd import hamiltonian as hm
from ad_afqmc_amd import propagation as pr
from ad_afqmc_amd import synthetic as syn
from ad_afqmc_amd import walkers as wk
from ad_afqmc_amd import wavefunctions as wf
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("e_est", [float("nan"), -3.0e5, 3.0e5, float("-inf")])
def test_weights_do_not_depend_on_e_estimate(e_est):
    print(f"[small shift] {e_est}", flush=True)
    n, o, g, w, dt = 10, 4, 20, 6, 0.01
    s = syn.make_system(n, o, g, seed=n, l_scale=2.0 / math.sqrt(n))
    trial = wf.rhf(n, (o, o))
    prop = pr.propagator_afqmc(dt=dt, n_walkers=w, n_exp_terms=6, walker_type="restricted")
    wave, ham, h = s.wave_data(), s.ham_data(), hm.hamiltonian(n)
    ham = h.build_measurement_intermediates(ham, trial, wave)
    ham = h.build_propagation_intermediates(ham, prop, trial, wave)
    h1, rh, rc = O.rhf_measurement_intermediates(s.h1, s.chol, s.mo_up)
    ot = O.RHFTrial(n, (o, o), s.mo_up)
    pi = O.propagation_intermediates(s.h0, h1, s.chol, s.rdm1(), dt, "restricted")
    oh = dict(h0=s.h0, chol=s.chol, rot_h1=rh, rot_chol=rc, **{k: pi[k] for k in ("mf_shifts", "h0_prop", "exp_h1")})
    up = syn.perturbed_walkers(s.mo_up, w, 0.05, 1)
    pd = prop.init_prop_data(trial, wave, ham, seed=0, init_walkers=wk.RHFWalkers(up))
    shift = float(pd["pop_control_ene_shift"].item())
    pd["e_estimate"] = e_est
    fields = np.random.default_rng(4).standard_normal((w, g))
    st = dict(walkers=up, weights=np.ones(w), overlaps=ot.calc_overlap(up), e_estimate=e_est,
              pop_control_ene_shift=shift)
    st = O.propagate_constrained(ot, st, fields, oh, dt, 6)
    assert np.all(st["weights"] > 0.1)
    new = prop.propagate_constrained(trial, ham, pd, fields, wave)
    got = new["weights"].cpu().numpy()
    assert np.max(np.abs(got - st["weights"])) < 1e-10 * np.max(st["weights"])
    left = float(new["pop_control_ene_shift"])
    ref = float(st["pop_control_ene_shift"])
    assert (math.isnan(ref) and math.isnan(left)) or left == ref or abs(left - ref) < 1e-10 * abs(ref)
