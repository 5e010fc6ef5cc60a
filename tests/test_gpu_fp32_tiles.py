"""FP32 Taylor terms of both spins' columns where the tile follows from the
padding: 48 x 80 tiles (67, 66 and 80 columns, rows of 48 k, one more and one
less) and 64 x 64 ones (128 columns, 64 k rows), against the oracle with the
tolerance of the FP32 mode."""
import math

import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, columns up, columns dn, W)
CASES = [(141, 35, 32, 3), (96, 40, 26, 2), (97, 41, 39, 2), (95, 33, 33, 9), (128, 64, 64, 2), (130, 64, 17, 1)]


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-c{c[1]}+{c[2]}" for c in CASES])
def test_fp32_propagator(case):
    n, cu, cd, w = case
    print(f"[fp32 tiles] {case}", flush=True)
    g, dt = 6, 0.01
    rng = np.random.default_rng(n)
    sysm = syn.make_system(n, cu, g, seed=n, l_scale=2.0 / math.sqrt(n))
    mo_dn = syn.make_system(n, cd, 1, seed=1).mo_up
    job = E.EngineJob(n, (cu, cd), g, w, "unrestricted", "uhf", 6, dt, "fp32")
    job.set_hamiltonian(0.0, sysm.h1, sysm.chol)
    job.set_trial(sysm.mo_up, mo_dn, sysm.rdm1())
    job.build_measurement()
    job.build_propagation()
    exp_h1 = np.stack([job.get(5, s).cpu().numpy() for s in range(2)])
    fields = rng.standard_normal((w, g)) + 0.3j * rng.standard_normal((w, g))
    walkers = [syn.perturbed_walkers(sysm.mo_up, w, 0.05, 1), syn.perturbed_walkers(mo_dn, w, 0.05, 2)]
    ref = O.apply_trotprop(walkers, fields, sysm.chol, exp_h1, dt, 6)
    dev = [torch.as_tensor(x).cuda() for x in walkers]
    job.trotprop(dev[0], dev[1], torch.as_tensor(fields).cuda())
    for a, b in zip(dev, ref):
        assert np.max(np.abs(a.cpu().numpy() - b)) < 2e-5 * np.max(np.abs(b))
