"""Set-up of the FP64 exchange's factors: for few occupied orbitals by one
work-group a Cholesky index (at its limits of 128 orbitals and 24 occupied, with
a chunk of Cholesky indices that is full, one short and one over, one spin on
each route), not at all for a job whose energies are formed without them, and
again for a new trial where rot_chol came from the caller.  Energies against the
oracle, 1e-10 of the largest, the repository's FP64 parity."""
import math

import numpy as np
import pytest

from ad_afqmc_amd import hamiltonian as hm
from ad_afqmc_amd import synthetic as syn
from ad_afqmc_amd import walkers as wk
from ad_afqmc_amd import wavefunctions as wf
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, O up, O dn or 0, G, W); 24 occupied: 5 Cholesky indices a tile, 16: 8, 7: 18
CASES = [(128, 24, 0, 10, 2), (127, 24, 23, 11, 3), (129, 24, 0, 9, 2), (96, 16, 0, 41, 3), (64, 7, 7, 36, 5),
         (64, 7, 6, 37, 2), (50, 25, 24, 30, 2), (90, 30, 3, 60, 2), (128, 1, 1, 300, 2), (24, 24, 0, 200, 2),
         (25, 24, 24, 190, 3), (100, 12, 11, 1, 2), (520, 20, 0, 3, 2)]


def _close(e, ref):
    return np.max(np.abs(e.cpu().numpy() - ref)) < 1e-10 * np.max(np.abs(ref))


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-O{c[1]}+{c[2]}-G{c[3]}" for c in CASES])
def test_energy(case):
    n, ou, od, g, w = case
    print(f"[exchange set-up] {case}", flush=True)
    uhf = od > 0
    s = syn.make_system(n, ou, g, nocc_dn=od or ou, uhf=uhf, seed=n + g, l_scale=2.0 / math.sqrt(n))
    trial = wf.uhf(n, (ou, od)) if uhf else wf.rhf(n, (ou, ou))
    wave = s.wave_data()
    ham = hm.hamiltonian(n).build_measurement_intermediates(s.ham_data(), trial, wave)
    up = syn.perturbed_walkers(s.mo_up, w, 0.3 / math.sqrt(n), seed=1)
    if uhf:
        dn = syn.perturbed_walkers(s.mo_dn, w, 0.3 / math.sqrt(n), seed=2)
        _, rh, rc = O.uhf_measurement_intermediates(s.h1, s.chol, s.mo_up, s.mo_dn)
        ref = O.UHFTrial(n, (ou, od), s.mo_up, s.mo_dn).calc_energy([up, dn], s.h0, rh, rc)
        e = trial.calc_energy(wk.UHFWalkers([up, dn]), ham, wave)
    else:
        _, rh, rc = O.rhf_measurement_intermediates(s.h1, s.chol, s.mo_up)
        ref = O.RHFTrial(n, (ou, ou), s.mo_up).calc_energy(up, s.h0, rh, rc)
        e = trial.calc_energy(wk.RHFWalkers(up), ham, wave)
    assert _close(e, ref)


@pytest.mark.parametrize("n,o,g", [(8, 3, 12), (30, 14, 40), (40, 18, 12)])
@pytest.mark.parametrize("supplied", [False, True])
def test_energy_follows_the_current_trial(n, o, g, supplied):
    """On one job, trial after trial, with rot_h1 and rot_chol built for each, or
    supplied by the caller once (the energy is then that of the arrays held)."""
    print(f"[exchange set-up] {n} {o} {g} {supplied}", flush=True)
    s = syn.make_system(n, o, g, seed=3, l_scale=2.0 / math.sqrt(n))
    walkers = syn.perturbed_walkers(s.mo_up, 4, 0.05, seed=1)
    wave, ham, trial = s.wave_data(), s.ham_data(), wf.rhf(n, (o, o))
    _, rh, rc = O.rhf_measurement_intermediates(s.h1, s.chol, s.mo_up)
    if supplied:
        ham.update(rot_h1=rh, rot_chol=rc)
    for seed in (0, 5, 7):
        if seed:
            mo = np.linalg.qr(s.mo_up + 0.05 * np.random.default_rng(seed).standard_normal((n, o)))[0]
            wave = dict(wave, mo_coeff=mo, rdm1=np.array([mo @ mo.T] * 2))
        mo = np.asarray(wave["mo_coeff"])
        if supplied:
            ham["rot_h1"] = rh.copy()
        else:
            ham = hm.hamiltonian(n).build_measurement_intermediates(ham, trial, wave)
            _, rh, rc = O.rhf_measurement_intermediates(s.h1, s.chol, mo)
        e = trial.calc_energy(wk.RHFWalkers(walkers), ham, wave)
        assert _close(e, O.RHFTrial(n, (o, o), mo).calc_energy(walkers, s.h0, rh, rc))
