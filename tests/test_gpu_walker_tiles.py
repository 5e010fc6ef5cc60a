"""The FP64 products over all walkers (VHS, force bias) in every instance that their
launchers choose, the full-height VHS tiles among them: walkers that leave the last
tile partly filled, contractions of a slab, one short and one over, on both sides of
the line between half and full height.  The instance that ran is read from the
kernel's name.  Some walkers of each case against the oracle: 1e-10 of the largest
value, the repository's FP64 parity."""
import math
import re

import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# instances: (row blocks, column blocks) of a wave, waves by rows and columns; (N, O up, O dn or 0, G, W, VHS instance)
FULL = {64: (4, 4, 2, 2), 32: (2, 2, 4, 2), 16: (2, 1, 4, 2)}
HALF = {64: (1, 4, 4, 2), 32: (1, 2, 4, 2), 16: (1, 1, 4, 2)}
CASES = [(220, 3, 0, 33, 130, FULL[64]), (222, 2, 2, 17, 65, FULL[64]), (290, 1, 0, 16, 33, FULL[64]),
         (300, 3, 2, 15, 63, FULL[64]), (290, 2, 0, 33, 17, FULL[32]), (279, 2, 1, 1, 31, FULL[32]),
         (290, 2, 0, 47, 5, FULL[16]), (275, 1, 1, 129, 16, FULL[16]), (304, 1, 0, 31, 1, FULL[16]),
         (272, 2, 0, 33, 64, HALF[64]), (257, 2, 1, 17, 65, FULL[64]), (260, 2, 0, 19, 20, HALF[32]),
         (271, 1, 0, 257, 9, HALF[16]), (100, 20, 19, 129, 70, HALF[64])]


def _kernels(call):
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    found = (re.search(r"walker_gemm_kernel<(\w+), (\d+), (\d+), (\d+), (\d+), (\w+)>", e.key) for e in p.key_averages())
    return [(m.group(6) == "true", tuple(int(m.group(i)) for i in (2, 3, 4, 5))) for m in found if m]


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-O{c[1]}+{c[2]}-G{c[3]}-W{c[4]}" for c in CASES])
def test_instance(case):
    n, ou, od, g, w, vhs = case
    print(f"[walker tiles] {case}", flush=True)
    dt, rng, uhf = 0.01, np.random.default_rng(n), od > 0
    sysm = syn.make_system(n, ou, g, seed=n, l_scale=2.0 / math.sqrt(n))
    mo_dn = syn.make_system(n, od, 1, seed=1).mo_up if uhf else None
    job = E.EngineJob(n, (ou, od or ou), g, w + 3, "unrestricted" if uhf else "restricted", "uhf" if uhf else "rhf", 2,
                      dt, "fp64")
    job.set_hamiltonian(0.0, sysm.h1, sysm.chol)
    job.set_trial(sysm.mo_up, mo_dn, sysm.rdm1())
    job.build_measurement()
    job.build_propagation()
    job.set_batch(w)
    walkers = [syn.perturbed_walkers(sysm.mo_up, w, 0.05, 1)] + ([syn.perturbed_walkers(mo_dn, w, 0.05, 2)] if uhf else [])
    dev = [torch.as_tensor(x).cuda() for x in walkers]
    pick = sorted({0, min(1, w - 1), w // 2, w - 1} | {w - w % 64 - 1} & set(range(w)))
    sub = [x[pick] for x in walkers]
    dn = dev[1] if uhf else None

    got = {}
    names = _kernels(lambda: got.update(fb=job.force_bias(dev[0], dn)))
    assert names == [(False, FULL[64 if w > 32 else 32 if w > 16 else 16])]
    if uhf:
        ref = O.UHFTrial(n, (ou, od), sysm.mo_up, mo_dn).calc_force_bias(
            sub, O.uhf_measurement_intermediates(sysm.h1, sysm.chol, sysm.mo_up, mo_dn)[2])
    else:
        ref = O.RHFTrial(n, (ou, ou), sysm.mo_up).calc_force_bias(
            sub[0], O.rhf_measurement_intermediates(sysm.h1, sysm.chol, sysm.mo_up)[2])
    fb = got["fb"].cpu().numpy()
    assert np.all(np.isfinite(fb)) and np.max(np.abs(fb[pick] - ref)) < 1e-10 * np.max(np.abs(ref))

    exp_h1 = np.stack([job.get(5, s).cpu().numpy() for s in range(2 if uhf else 1)])
    fields = rng.standard_normal((w, g)) + 0.3j * rng.standard_normal((w, g))
    f = torch.as_tensor(fields).cuda()
    assert _kernels(lambda: job.trotprop(dev[0], dn, f)) == [(True, vhs)]
    ref = O.apply_trotprop(sub if uhf else sub[0], fields[pick], sysm.chol, exp_h1 if uhf else exp_h1[0], dt, 2)
    for a, b in zip(dev, ref if uhf else [ref]):
        a = a.cpu().numpy()
        assert np.all(np.isfinite(a)) and np.max(np.abs(a[pick] - b)) < 1e-10 * np.max(np.abs(b))
