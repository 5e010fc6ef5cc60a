"""The FP64 exchange's walker-independent part with trials whose orbitals are far
from orthonormal (condition 1e3 to 1e5): T = T0 A spans what T0 spans, and every
energy is that of T0.  The engine may be no further off than the plain formula
f = rot_chol G^T is in FP64, in geometric mean over 18 systems, against T0 in
extended precision; the error itself varies from system to system by 3 or so."""
import math

import numpy as np
import pytest

from ad_afqmc_amd import hamiltonian as hm
from ad_afqmc_amd import walkers as wk
from ad_afqmc_amd import wavefunctions as wf

pytestmark = pytest.mark.gpu


def _inverse(s):
    """Gauss-Jordan with partial pivoting in s's own type."""
    n = s.shape[0]
    a = np.concatenate([s, np.eye(n, dtype=s.dtype)], 1)
    for k in range(n):
        p = k + np.argmax(np.abs(a[k:, k]))
        a[[k, p]] = a[[p, k]]
        a[k] /= a[k, k]
        for i in range(n):
            if i != k:
                a[i] -= a[i, k] * a[k]
    return a[:, n:]


def _energies(h1, chol, t, walkers, real):
    cplx = np.result_type(real, 1j)
    n, t = h1.shape[0], t.astype(real)
    rc = t.T @ chol.reshape(-1, n, n).astype(real)
    out = []
    for w in walkers.astype(cplx):
        gt = w @ _inverse(t.T.astype(cplx) @ w)
        f = rc @ gt
        e = 2 * np.trace(t.T @ h1.astype(real) @ gt)
        out.append(e + 2 * np.sum(np.trace(f, axis1=1, axis2=2) ** 2) - np.sum(f * f.transpose(0, 2, 1)))
    return np.array(out)


def test_energies_of_trials_far_from_orthonormal():
    n, o, g, w = 40, 20, 12, 16
    logs = []
    for seed in range(6):
        rng = np.random.default_rng(seed)
        chol = 0.2 * rng.standard_normal((g, n, n))
        chol = ((chol + chol.transpose(0, 2, 1)) / 2).reshape(g, n * n)
        h1 = np.diag(np.linspace(-2.0, 1.0, n))
        t0 = np.linalg.qr(rng.standard_normal((n, o)))[0]
        walkers = t0 + 0.1 * (rng.standard_normal((w, n, o)) + 1j * rng.standard_normal((w, n, o)))
        ref = _energies(h1, chol, t0, walkers, np.longdouble)
        for k in (3, 4, 5):
            u, v = (np.linalg.qr(rng.standard_normal((o, o)))[0] for _ in range(2))
            t = t0 @ (u * np.logspace(0, -k, o)) @ v.T
            trial = wf.rhf(n, (o, o))
            wave = {"mo_coeff": t, "rdm1": np.array([t0 @ t0.T] * 2)}
            ham = {"h0": 0.0, "h1": np.array([h1, h1]), "chol": chol}
            ham = hm.hamiltonian(n).build_measurement_intermediates(ham, trial, wave)
            e = trial.calc_energy(wk.RHFWalkers(walkers), ham, wave).cpu().numpy()
            rms = [float(np.sqrt(np.mean(np.abs((x - ref).astype(np.complex128)) ** 2))) for x in
                   (e, _energies(h1, chol, t, walkers, np.float64))]
            print(f"[trial] seed {seed} condition 1e{k}: engine {rms[0]:.1e}, plain {rms[1]:.1e}", flush=True)
            logs.append(math.log(rms[0] / rms[1]))
    assert math.exp(np.mean(logs)) <= 1.0
