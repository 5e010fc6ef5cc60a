"""Energies over the numbers of walkers at which the FP64 exchange changes: few
ones (theta of both spins in one launch, tiles narrowed to the walkers or until
they fill the chip, two and three row blocks a wave, small jobs among them, and a
batch below the job's capacity), and past them, where theta is a product of its
own.  Against the oracle, 1e-10 of the largest, the repository's FP64 parity."""
import math

import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, O up, O dn or 0, G, walkers of the job, walkers measured)
CASES = [(110, 16, 0, 9, 5, 1), (110, 16, 0, 9, 5, 3), (110, 16, 15, 70, 9, 5), (400, 5, 0, 39, 20, 3),
         (400, 5, 4, 77, 9, 9), (140, 12, 0, 33, 12, 2), (60, 24, 0, 17, 7, 1), (60, 24, 23, 17, 7, 3),
         (61, 20, 17, 13, 7, 2), (80, 25, 19, 6, 6, 1), (80, 32, 31, 9, 4, 2), (90, 40, 33, 7, 3, 3),
         (130, 64, 65, 3, 2, 2), (140, 97, 1, 3, 2, 1), (48, 16, 16, 60, 40, 7), (60, 12, 11, 50, 3, 2),
         (37, 9, 7, 300, 30, 30), (30, 17, 0, 2, 700, 700), (17, 17, 17, 5, 3, 2), (66, 66, 0, 3, 2, 2),
         (140, 12, 0, 33, 180, 180),
         # past the few
         (300, 60, 58, 3, 34, 33), (260, 97, 0, 2, 33, 31), (250, 33, 20, 3, 160, 65), (250, 34, 33, 2, 71, 70),
         (76, 16, 15, 9, 3, 3), (75, 16, 16, 9, 3, 2), (150, 16, 0, 9, 3, 2)]


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-O{c[1]}+{c[2]}-G{c[3]}-W{c[5]}of{c[4]}" for c in CASES])
def test_energy(case):
    n, ou, od, g, cap, w = case
    print(f"[exchange walkers] {case}", flush=True)
    uhf = od > 0
    s = syn.make_system(n, ou, g, seed=n + w, l_scale=2.0 / math.sqrt(n))
    mo_dn = syn.make_system(n, od, 1, seed=1).mo_up if uhf else None
    job = E.EngineJob(n, (ou, od or ou), g, cap, "unrestricted" if uhf else "restricted", "uhf" if uhf else "rhf", 2,
                      0.01, "fp64")
    job.set_hamiltonian(s.h0, s.h1, s.chol)
    job.set_trial(s.mo_up, mo_dn, s.rdm1())
    job.build_measurement()
    amp = 0.3 / math.sqrt(n)
    walkers = [syn.perturbed_walkers(s.mo_up, w, amp, 1)] + ([syn.perturbed_walkers(mo_dn, w, amp, 2)] if uhf else [])
    dev = [torch.as_tensor(x).cuda() for x in walkers]
    job.set_batch(w)
    e = job.energy(dev[0], dev[1] if uhf else None).cpu().numpy()
    pick = sorted({0, w // 2, w - 1} | set(range(min(w, 6))))  # walkers are independent
    if uhf:
        _, rh, rc = O.uhf_measurement_intermediates(s.h1, s.chol, s.mo_up, mo_dn)
        ref = O.UHFTrial(n, (ou, od), s.mo_up, mo_dn).calc_energy([x[pick] for x in walkers], s.h0, rh, rc)
    else:
        _, rh, rc = O.rhf_measurement_intermediates(s.h1, s.chol, s.mo_up)
        ref = O.RHFTrial(n, (ou, ou), s.mo_up).calc_energy(walkers[0][pick], s.h0, rh, rc)
    assert np.all(np.isfinite(e))
    assert np.max(np.abs(e[pick] - ref)) < 1e-10 * np.max(np.abs(ref))
