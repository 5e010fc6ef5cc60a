"""The FP64 products over all walkers (force bias, VHS) at the edges of their
tiles: walkers around 16, 32 and 64, odd and short contractions, Cholesky counts
around 128, one and two spins, slices that do not fill.  Against the oracle,
1e-10 of the largest value, the repository's FP64 parity."""
import math

import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, O up, O dn or 0, G, W, walkers the job is made for)
CASES = [(50, 17, 0, 129, 1, 1), (51, 9, 7, 128, 16, 16), (49, 1, 1, 200, 17, 40), (57, 19, 18, 127, 33, 33),
         (64, 20, 20, 1, 64, 64), (75, 3, 0, 255, 65, 65), (81, 41, 39, 17, 31, 31), (113, 5, 33, 300, 70, 128),
         (97, 30, 29, 1000, 2, 2)]


def _rel(a, b):
    return np.max(np.abs(a - b)) / np.max(np.abs(b))


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-O{c[1]}+{c[2]}-G{c[3]}-W{c[4]}" for c in CASES])
def test_products_at_tile_edges(case):
    n, ou, od, g, w, cap = case
    print(f"[products] {case}", flush=True)
    dt = 0.01
    rng = np.random.default_rng(n)
    sysm = syn.make_system(n, ou, g, seed=n, l_scale=2.0 / math.sqrt(n))
    uhf = od > 0
    job = E.EngineJob(n, (ou, od or ou), g, cap, "unrestricted" if uhf else "restricted", "uhf" if uhf else "rhf", 2,
                      dt, "fp64")
    mo_dn = syn.make_system(n, od, 1, seed=1).mo_up if uhf else None
    job.set_hamiltonian(0.0, sysm.h1, sysm.chol)
    job.set_trial(sysm.mo_up, mo_dn, sysm.rdm1())
    job.build_measurement()
    job.build_propagation()
    up = syn.perturbed_walkers(sysm.mo_up, w, 0.05, 1)
    walkers = [up, syn.perturbed_walkers(mo_dn, w, 0.05, 2)] if uhf else up
    dev = [torch.as_tensor(x).cuda() for x in (walkers if uhf else [walkers])]
    job.set_batch(w)

    if uhf:
        fb = O.UHFTrial(n, (ou, od), sysm.mo_up, mo_dn).calc_force_bias(
            walkers, O.uhf_measurement_intermediates(sysm.h1, sysm.chol, sysm.mo_up, mo_dn)[2])
    else:
        fb = O.RHFTrial(n, (ou, ou), sysm.mo_up).calc_force_bias(
            walkers, O.rhf_measurement_intermediates(sysm.h1, sysm.chol, sysm.mo_up)[2])
    assert _rel(job.force_bias(dev[0], dev[1] if uhf else None).cpu().numpy(), fb) < 1e-10

    exp_h1 = np.stack([job.get(5, s).cpu().numpy() for s in range(2 if uhf else 1)])
    fields = rng.standard_normal((w, g)) + 0.3j * rng.standard_normal((w, g))
    ref = O.apply_trotprop(walkers, fields, sysm.chol, exp_h1 if uhf else exp_h1[0], dt, 2)
    job.trotprop(dev[0], dev[1] if uhf else None, torch.as_tensor(fields).cuda())
    for a, b in zip(dev, ref if uhf else [ref]):
        assert _rel(a.cpu().numpy(), b) < 1e-10
