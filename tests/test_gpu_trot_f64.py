"""The fused FP64 propagator at the edges of its tiles (one row block more or
less than eight waves take, column blocks split over waves, slabs of one column
block and a last one that is partly filled, both spins, one and two Taylor
terms), against the oracle: 1e-10 of the largest value, the repository's FP64
parity."""
import math

import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, columns up, columns dn or 0, W, Taylor terms)
CASES = [(49, 17, 0, 3, 6), (64, 20, 18, 9, 6), (80, 8, 0, 17, 1), (112, 33, 0, 2, 2), (129, 24, 23, 5, 6),
         (176, 41, 0, 8, 6), (208, 1, 1, 2, 6), (241, 40, 0, 3, 6), (304, 60, 58, 2, 6), (400, 33, 0, 2, 6),
         (512, 9, 0, 1, 6), (624, 20, 0, 1, 3), (650, 12, 0, 1, 3)]


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-c{c[1]}+{c[2]}-K{c[4]}" for c in CASES])
def test_propagator_at_tile_edges(case):
    n, cu, cd, w, terms = case
    print(f"[trot] {case}", flush=True)
    g, dt = 6, 0.01
    rng = np.random.default_rng(n)
    sysm = syn.make_system(n, cu, g, seed=n, l_scale=2.0 / math.sqrt(n))
    uhf = cd > 0
    job = E.EngineJob(n, (cu, cd or cu), g, w, "unrestricted" if uhf else "restricted", "uhf" if uhf else "rhf", terms,
                      dt, "fp64")
    mo_dn = syn.make_system(n, cd, 1, seed=1).mo_up if uhf else None
    job.set_hamiltonian(0.0, sysm.h1, sysm.chol)
    job.set_trial(sysm.mo_up, mo_dn, sysm.rdm1())
    job.build_measurement()
    job.build_propagation()
    exp_h1 = np.stack([job.get(5, s).cpu().numpy() for s in range(2 if uhf else 1)])
    fields = rng.standard_normal((w, g)) + 0.3j * rng.standard_normal((w, g))
    up = syn.perturbed_walkers(sysm.mo_up, w, 0.05, 1)
    walkers = [up, syn.perturbed_walkers(mo_dn, w, 0.05, 2)] if uhf else up
    ref = O.apply_trotprop(walkers, fields, sysm.chol, exp_h1 if uhf else exp_h1[0], dt, terms)
    dev = [torch.as_tensor(x).cuda() for x in (walkers if uhf else [walkers])]
    job.trotprop(dev[0], dev[1] if uhf else None, torch.as_tensor(fields).cuda())
    for a, b in zip(dev, ref if uhf else [ref]):
        assert np.max(np.abs(a.cpu().numpy() - b)) < 1e-10 * np.max(np.abs(b))
