"""FP64 exchange over the trial's unoccupied orbitals, at the edges of its tiles
(one more or less than a multiple of 16 occupied orbitals, one wave column and
whole f blocks, several walkers a tile and a last group of fewer, d kept whole
or in strips, no unoccupied orbital at all), against the oracle.  1e-10 of the
largest energy, the repository's FP64 parity."""
import math

import numpy as np
import pytest

from ad_afqmc_amd import hamiltonian as hm
from ad_afqmc_amd import synthetic as syn
from ad_afqmc_amd import walkers as wk
from ad_afqmc_amd import wavefunctions as wf
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, nocc, G, W): nocc > 16 keeps clear of the one-work-group measurement
CASES = [(18, 17, 3, 7), (33, 24, 17, 5), (40, 33, 9, 3), (64, 48, 5, 2), (70, 49, 11, 2), (71, 53, 6, 3),
         (66, 64, 5, 2), (80, 65, 5, 2), (100, 96, 4, 2), (99, 97, 3, 2), (140, 128, 3, 1), (132, 129, 3, 1),
         (20, 20, 4, 3), (97, 97, 2, 2)]


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-O{c[1]}" for c in CASES])
@pytest.mark.parametrize("skew", [False, True], ids=["orthonormal", "skewed"])
def test_energy_at_tile_edges(case, skew):
    n, o, g, w = case
    print(f"[exchange] {case} skew={skew}", flush=True)
    s = syn.make_system(n, o, g, seed=o, l_scale=2.0 / math.sqrt(n))
    mo = s.mo_up
    if skew:  # a trial whose orbitals are neither normalised nor orthogonal
        mo = mo @ (np.eye(o) + 0.2 / math.sqrt(o) * np.random.default_rng(o).standard_normal((o, o)))
    trial = wf.rhf(n, (o, o))
    wave = {"mo_coeff": mo, "rdm1": np.array([mo @ mo.T] * 2)}
    ham = hm.hamiltonian(n).build_measurement_intermediates(s.ham_data(), trial, wave)
    walkers = syn.perturbed_walkers(mo, w, 0.3 / math.sqrt(n), seed=1)
    e = trial.calc_energy(wk.RHFWalkers(walkers), ham, wave).cpu().numpy()
    _, rh, rc = O.rhf_measurement_intermediates(s.h1, s.chol, mo)
    ref = O.RHFTrial(n, (o, o), mo).calc_energy(walkers, s.h0, rh, rc)
    assert np.max(np.abs(e - ref)) < 1e-10 * np.max(np.abs(ref))


def test_energy_follows_the_current_trial():
    """rot_chol supplied by the caller, then another trial: the energy is that
    of the walkers with the new trial and the arrays now held."""
    n, o, g, w = 30, 18, 12, 4
    s = syn.make_system(n, o, g, seed=3, l_scale=2.0 / math.sqrt(n))
    walkers = syn.perturbed_walkers(s.mo_up, w, 0.05, seed=1)
    _, rh, rc = O.rhf_measurement_intermediates(s.h1, s.chol, s.mo_up)
    wave, ham = s.wave_data(), dict(s.ham_data(), rot_h1=rh, rot_chol=rc)
    trial = wf.rhf(n, (o, o))
    for seed in (0, 5):
        if seed:
            mo = np.linalg.qr(s.mo_up + 0.05 * np.random.default_rng(seed).standard_normal((n, o)))[0]
            wave["mo_coeff"], wave["rdm1"] = mo, np.array([mo @ mo.T] * 2)
            ham["rot_h1"] = rh.copy()  # a new trial needs one of the intermediates set again; rot_chol stays
        e = trial.calc_energy(wk.RHFWalkers(walkers), ham, wave).cpu().numpy()
        ref = O.RHFTrial(n, (o, o), np.asarray(wave["mo_coeff"])).calc_energy(walkers, s.h0, rh, rc)
        assert np.max(np.abs(e - ref)) < 1e-10 * np.max(np.abs(ref))
