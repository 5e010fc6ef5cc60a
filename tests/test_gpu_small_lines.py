"""Small FP64 jobs on both sides of the line up to which their steps run in one
work-group a walker: bytes of L and rot_chol a CU, 2.5 MB where L is packed and 9.5
where it is not, just below and just above by Cholesky vectors and by walkers (256 and
257).  A step against the oracle on some walkers, 1e-10 of the largest value, the
repository's FP64 parity; the path is read from the kernels that ran."""
import math

import numpy as np
import pytest
import torch

from ad_afqmc_amd import hamiltonian as hm
from ad_afqmc_amd import propagation as pr
from ad_afqmc_amd import synthetic as syn
from ad_afqmc_amd import walkers as wk
from ad_afqmc_amd import wavefunctions as wf
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, O up = O dn, G, W, antisymmetric part of L, one work-group a walker)
CASES = [(48, 16, 115, 5, 0.0, True), (48, 16, 116, 5, 0.0, False), (48, 9, 76, 256, 0.0, True),
         (48, 9, 77, 257, 0.0, False), (40, 10, 494, 3, 0.0, True), (40, 10, 495, 3, 0.0, False),
         (30, 8, 430, 257, 0.0, True), (30, 8, 431, 257, 0.0, False), (48, 9, 374, 2, 1e-3, True),
         (48, 9, 375, 2, 1e-3, False)]


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-O{c[1]}-G{c[2]}-W{c[3]}-{c[4]}" for c in CASES])
def test_step(case):
    n, o, g, w, asym, small = case
    print(f"[small lines] {case}", flush=True)
    dt = 0.01
    s = syn.make_system(n, o, g, nocc_dn=o, uhf=True, seed=n, l_scale=2.0 / math.sqrt(n))
    if asym:
        a = np.random.default_rng(n).standard_normal((g, n, n))
        s.chol += asym / math.sqrt(g) * (a - a.transpose(0, 2, 1)).reshape(g, n * n)
    trial = wf.uhf(n, (o, o))
    prop = pr.propagator_afqmc(dt=dt, n_walkers=w, n_exp_terms=6, walker_type="unrestricted")
    wave, ham, h = s.wave_data(), s.ham_data(), hm.hamiltonian(n)
    ham = h.build_measurement_intermediates(ham, trial, wave)
    ham = h.build_propagation_intermediates(ham, prop, trial, wave)
    ot = O.UHFTrial(n, (o, o), s.mo_up, s.mo_dn)
    h1, rh, rc = O.uhf_measurement_intermediates(s.h1, s.chol, s.mo_up, s.mo_dn)
    pi = O.propagation_intermediates(s.h0, h1, s.chol, s.rdm1(), dt, "unrestricted")
    oh = dict(h0=s.h0, chol=s.chol, rot_h1=rh, rot_chol=rc, **{k: pi[k] for k in ("mf_shifts", "h0_prop", "exp_h1")})
    walkers = [syn.perturbed_walkers(m, w, 0.3 / math.sqrt(n), i) for i, m in enumerate((s.mo_up, s.mo_dn))]
    pd = prop.init_prop_data(trial, wave, ham, seed=0, init_walkers=wk.UHFWalkers(walkers))
    fields = np.random.default_rng(4).standard_normal((w, g))
    out = {}
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
        out.update(prop.propagate_constrained(trial, ham, pd, fields, wave))
        torch.cuda.synchronize()
    assert any("small_step_kernel" in e.key for e in p.key_averages()) == small
    pick = sorted({0, min(1, w - 1), w // 2, w - 1})
    shift = float(pd["pop_control_ene_shift"])
    sub = [x[pick] for x in walkers]
    st = dict(walkers=sub, weights=np.ones(len(pick)), overlaps=ot.calc_overlap(sub),
              e_estimate=float(pd["e_estimate"]), pop_control_ene_shift=shift)
    st = O.propagate_constrained(ot, st, fields[pick], oh, dt, 6)
    for a, b in [(out["weights"], st["weights"]), (out["overlaps"], st["overlaps"])] + list(
            zip(out["walkers"].tensors(), st["walkers"])):
        a = a.cpu().numpy()
        assert np.all(np.isfinite(a)) and np.max(np.abs(a[pick] - b)) < 1e-10 * np.max(np.abs(b))
