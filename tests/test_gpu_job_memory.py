"""A job's small buffers lie in pieces below 2 MB and its large ones in one
allocation, or above 48 MB all in one: jobs without large buffers, with both and
past that line give the oracle's step and energy (each buffer in a place of its
own; 1e-10 of the largest value, the repository's FP64 parity), and creating and
closing them over and over leaves no memory behind."""
import ctypes as C
import math

import numpy as np
import pytest
import torch

from ad_afqmc_amd import _native as nat
from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, O, G, W): 3, 15, 33, 47 and 53 MB of buffers
CASES = [(20, 5, 40, 40), (30, 17, 120, 64), (48, 16, 160, 64), (48, 16, 200, 80), (60, 20, 240, 64)]


def _megabytes(n, o, g, w):
    d = nat.JobDesc(norb=n, nelec_up=o, nelec_dn=o, nchol=g, n_walkers=w, walker_type=nat.AFQ_WALKERS_RESTRICTED,
                    trial_type=nat.AFQ_TRIAL_RHF, n_exp_terms=6, precision=nat.PRECISIONS["fp64"], reserved=0, dt=0.01)
    return nat.lib().afq_job_footprint(C.byref(d), 0) / 1e6


def _job(s, n, o, g, w):
    job = E.EngineJob(n, (o, o), g, w, "restricted", "rhf", 6, 0.01, "fp64")
    job.set_hamiltonian(0.0, s.h1, s.chol)
    job.set_trial(s.mo_up, None, s.rdm1())
    job.build_measurement()
    job.build_propagation()
    return job


def test_sizes_lie_on_both_sides():
    sizes = [_megabytes(*c) for c in CASES]
    assert min(sizes) < 16 < 48 < max(sizes) and any(16 < x < 48 for x in sizes)


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-W{c[3]}" for c in CASES])
def test_results_and_memory(case):
    n, o, g, w = case
    print(f"[job memory] {case}", flush=True)
    s = syn.make_system(n, o, g, seed=n, l_scale=2.0 / math.sqrt(n))
    up = syn.perturbed_walkers(s.mo_up, w, 0.05, 1)
    h1, rh, rc = O.rhf_measurement_intermediates(s.h1, s.chol, s.mo_up)
    ot = O.RHFTrial(n, (o, o), s.mo_up)
    pi = O.propagation_intermediates(0.0, h1, s.chol, s.rdm1(), 0.01)
    fields = np.random.default_rng(n).standard_normal((w, g))
    st = dict(walkers=up, weights=np.ones(w), overlaps=ot.calc_overlap(up), e_estimate=-1.0, pop_control_ene_shift=-1.0)
    ham = dict(chol=s.chol, rot_chol=rc, **{k: pi[k] for k in ("mf_shifts", "h0_prop", "exp_h1")})
    st = O.propagate_constrained(ot, st, fields, ham, 0.01, 6)
    e_ref = ot.calc_energy(st["walkers"], 0.0, rh, rc)
    free = None
    for _ in range(6):
        job = _job(s, n, o, g, w)
        dev = torch.as_tensor(up).cuda()
        weights = torch.ones(w, dtype=torch.float64, device="cuda")
        overlaps = job.overlap(dev, None)
        scalars = torch.tensor([-1.0, -1.0], dtype=torch.float64, device="cuda")
        job.propagate(dev, None, torch.as_tensor(fields).cuda(), weights, overlaps, scalars, None)
        for a, b in ((dev, st["walkers"]), (weights, st["weights"]), (overlaps, st["overlaps"]),
                     (job.energy(dev, None), e_ref)):
            assert np.max(np.abs(a.cpu().numpy() - b)) < 1e-10 * np.max(np.abs(b))
        job.close()
        now = torch.cuda.mem_get_info()[0]
        free = free if free is not None else now
    assert free - now < 16 << 20
