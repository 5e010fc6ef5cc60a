"""Small FP64 jobs, whose steps and measurements run in one work-group per
walker: at the limits of that path (48 orbitals, 16 occupied per spin), with L
resident and streamed, at the smallest sizes, and past the limits, against the
oracle.  1e-10 of each quantity's largest value, the repository's FP64 parity."""
import math

import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import hamiltonian as hm
from ad_afqmc_amd import propagation as pr
from ad_afqmc_amd import synthetic as syn
from ad_afqmc_amd import walkers as wk
from ad_afqmc_amd import wavefunctions as wf
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (trial, walkers, N, nocc_up, nocc_dn, G, W, Taylor terms, antisymmetric part of L)
CASES = [("rhf", "restricted", 2, 1, 1, 1, 1, 6, 0.0), ("rhf", "restricted", 4, 4, 4, 5, 3, 6, 0.0),
         ("rhf", "restricted", 10, 5, 5, 27, 50, 6, 0.0), ("uhf", "restricted", 17, 9, 6, 33, 5, 6, 0.0),
         ("rhf", "unrestricted", 16, 8, 8, 40, 300, 6, 0.0), ("uhf", "unrestricted", 37, 13, 12, 149, 9, 6, 0.0),
         ("uhf", "unrestricted", 48, 16, 16, 60, 4, 6, 0.0), ("rhf", "restricted", 48, 16, 16, 130, 3, 2, 1e-3),
         ("rhf", "restricted", 13, 3, 3, 20, 6, 1, 1e-3), ("rhf", "restricted", 49, 16, 16, 60, 4, 6, 0.0),
         ("uhf", "unrestricted", 30, 17, 16, 60, 4, 6, 0.0), ("rhf", "restricted", 90, 16, 16, 50, 5, 6, 0.0)]
IDS = [f"{c[0]}-{c[1]}-N{c[2]}-O{c[3]}-K{c[7]}" for c in CASES]


def _rel(a, b):
    a, b = (x.detach().cpu().numpy() if isinstance(x, torch.Tensor) else np.asarray(x) for x in (a, b))
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def _setup(kind, wtype, n, ou, od, g, w, terms, asym, dt=0.01):
    s = syn.make_system(n, ou, g, nocc_dn=od, uhf=kind == "uhf", seed=n, l_scale=min(1.0, 2.0 / math.sqrt(n)))
    if asym:
        a = np.random.default_rng(n).standard_normal((g, n, n))
        s.chol += asym * (a - a.transpose(0, 2, 1)).reshape(g, n * n)
    trial = wf.rhf(n, (ou, ou)) if kind == "rhf" else wf.uhf(n, (ou, od))
    prop = pr.propagator_afqmc(dt=dt, n_walkers=w, n_exp_terms=terms, walker_type=wtype)
    wave, ham, h = s.wave_data(), s.ham_data(), hm.hamiltonian(n)
    ham = h.build_measurement_intermediates(ham, trial, wave)
    ham = h.build_propagation_intermediates(ham, prop, trial, wave)
    if kind == "rhf":
        h1, rh, rc = O.rhf_measurement_intermediates(s.h1, s.chol, s.mo_up)
        ot = O.RHFTrial(n, (ou, ou), s.mo_up)
    else:
        h1, rh, rc = O.uhf_measurement_intermediates(s.h1, s.chol, s.mo_up, s.mo_dn)
        ot = O.UHFTrial(n, (ou, od), s.mo_up, s.mo_dn)
    pi = O.propagation_intermediates(s.h0, h1, s.chol, s.rdm1(), dt, wtype)
    oh = dict(h0=s.h0, chol=s.chol, rot_h1=rh, rot_chol=rc, **{k: pi[k] for k in ("mf_shifts", "h0_prop", "exp_h1")})
    up = syn.perturbed_walkers(s.mo_up, w, 0.3 / math.sqrt(n), 1)
    if wtype == "restricted":
        return trial, prop, wave, ham, ot, oh, wk.RHFWalkers(up), up
    dn = syn.perturbed_walkers(s.mo_up if s.mo_dn is None else s.mo_dn, w, 0.3 / math.sqrt(n), 2)
    return trial, prop, wave, ham, ot, oh, wk.UHFWalkers([up, dn]), [up, dn]


@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_step_and_measurement(case):
    print(f"[small] {case}", flush=True)
    trial, prop, wave, ham, ot, oh, w, ow = _setup(*case)
    dt, terms, n_w = prop.dt, case[7], case[6]
    pd = prop.init_prop_data(trial, wave, ham, seed=0, init_walkers=w)
    assert _rel(pd["overlaps"], ot.calc_overlap(ow)) < 1e-10
    e_ref = ot.calc_energy(ow, oh["h0"], oh["rot_h1"], oh["rot_chol"])
    assert _rel(trial.calc_energy(w, ham, wave), e_ref) < 1e-10
    fields = np.random.default_rng(4).standard_normal((n_w, case[5]))
    e_est = float(pd["e_estimate"].item())
    st = dict(walkers=ow, weights=np.ones(n_w), overlaps=ot.calc_overlap(ow), e_estimate=e_est,
              pop_control_ene_shift=e_est)
    st = O.propagate_constrained(ot, st, fields, oh, dt, terms)
    new = prop.propagate_constrained(trial, ham, pd, fields, wave, return_force_bias=True)
    assert _rel(new["force_bias"], st["force_bias"]) < 1e-10
    assert _rel(new["overlaps"], st["overlaps"]) < 1e-10
    assert _rel(new["weights"], st["weights"]) < 1e-10
    assert _rel(new["pop_control_ene_shift"], st["pop_control_ene_shift"]) < 1e-10
    for a, b in zip(new["walkers"].tensors(), [st["walkers"], None] if w.tensors()[1] is None else st["walkers"]):
        if a is not None:
            assert _rel(a, b) < 1e-10


@pytest.mark.parametrize("case", [CASES[2], CASES[5], CASES[9]], ids=[IDS[2], IDS[5], IDS[9]])
def test_block_equals_its_steps(case):
    """A block (its steps in one launch) against the steps one by one, the QR,
    the energies and the block's bookkeeping with the same fields."""
    print(f"[small block] {case}", flush=True)
    trial, prop, wave, ham, ot, oh, w, ow = _setup(*case)
    g, n_w, steps, seed = case[5], case[6], 4, 11
    job = prop._job(trial, ham, wave, n_w)
    pd = prop.init_prop_data(trial, wave, ham, seed=0, init_walkers=w)
    up, dn = (None if t is None else t.clone() for t in w.tensors())
    weights, overlaps = torch.linspace(0.5, 1.5, n_w, dtype=torch.float64, device="cuda"), pd["overlaps"].clone()
    e = pd["e_estimate"]
    scalars = torch.stack([e, e]).contiguous()
    fields = E.normal_fill(steps * n_w * g, seed, 3).reshape(steps, n_w, g)
    ref = dict(pd, weights=weights.clone())
    for f in fields:
        ref = prop.propagate_constrained(trial, ham, ref, f, wave)
    out, _ = job.block(up, dn, weights, overlaps, scalars, steps, seed, 3)
    assert _rel(weights, ref["weights"]) < 1e-10
    q = ref["walkers"].orthonormalize()
    for a, b in zip((up, dn), q.tensors()):
        if a is not None:
            assert _rel(a, b) < 1e-10
    assert _rel(overlaps, trial.calc_overlap(q, wave)) < 1e-10
    energy = trial.calc_energy(q, ham, wave).real
    energy = torch.where((energy - e).abs() > math.sqrt(2.0 / prop.dt), e, energy)  # the block's energy window
    mean = (energy * ref["weights"]).sum() / ref["weights"].sum()
    assert _rel(out, torch.stack([mean, ref["weights"].sum()])) < 1e-10
    assert _rel(scalars[1], 0.9 * ref["pop_control_ene_shift"] + 0.1 * mean) < 1e-10
