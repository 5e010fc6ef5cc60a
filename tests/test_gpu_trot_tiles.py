"""The fused FP64 propagator in every instance that its launcher can choose: row
blocks a wave, column blocks a slab (the last slab partly filled) and column-split
blocks, one and two spins, up to its last size (560 orbitals) and one past it.  The
instance that ran is read from the kernel's name, so that a change of the rule
which leaves one without a case is seen.  Some walkers of each case against the
oracle: 1e-10 of the largest value, the repository's FP64 parity."""
import math
import re

import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, columns up, columns dn or 0, W, (row blocks, column blocks, column-split blocks) of a wave)
CASES = [(32, 17, 0, 3, (1, 2, 1)), (48, 20, 17, 2, (1, 1, 1)), (61, 1, 0, 1, (1, 1, 0)), (69, 1, 0, 1, (1, 1, 1)),
         (61, 29, 26, 33, (1, 2, 0)), (69, 29, 26, 33, (1, 2, 1)), (61, 49, 46, 40, (1, 3, 0)),
         (69, 21, 18, 65, (1, 3, 1)), (97, 49, 46, 40, (1, 3, 2)), (61, 29, 26, 100, (1, 4, 0)),
         (69, 29, 26, 65, (1, 4, 1)), (97, 29, 26, 100, (1, 4, 2)), (61, 33, 0, 230, (1, 5, 0)),
         (69, 37, 34, 90, (1, 5, 1)), (81, 37, 34, 90, (1, 5, 2)), (177, 1, 0, 1, (2, 1, 0)),
         (193, 1, 0, 1, (2, 1, 1)), (177, 29, 26, 33, (2, 2, 0)), (193, 29, 26, 33, (2, 2, 1)),
         (177, 49, 46, 40, (2, 3, 0)), (193, 49, 46, 40, (2, 3, 1)), (225, 49, 46, 40, (2, 3, 2)),
         (177, 29, 26, 100, (2, 4, 0)), (193, 29, 26, 100, (2, 4, 1)), (225, 29, 26, 100, (2, 4, 2)),
         (177, 33, 0, 230, (2, 5, 0)), (193, 33, 0, 230, (2, 5, 1)), (209, 33, 0, 230, (2, 5, 2)),
         (305, 1, 0, 1, (3, 1, 0)), (321, 9, 0, 2, (3, 1, 1)), (305, 29, 26, 33, (3, 2, 0)),
         (321, 29, 26, 33, (3, 2, 1)), (305, 49, 46, 40, (3, 3, 0)), (321, 49, 46, 40, (3, 3, 1)),
         (353, 49, 46, 40, (3, 3, 2)), (433, 5, 0, 1, (4, 1, 0)), (449, 9, 0, 2, (4, 1, 1)),
         (433, 29, 26, 33, (4, 2, 0)), (449, 29, 26, 33, (4, 2, 1)), (513, 9, 0, 1, (4, 1, 1)),
         (545, 12, 9, 2, (4, 1, 1)), (560, 29, 26, 33, (4, 2, 1))]


def _kernels(call):
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    return [e.key for e in p.key_averages()]


def _run(n, cu, cd, w):
    g, dt, terms = 3, 0.01, 4
    rng = np.random.default_rng(n)
    sysm = syn.make_system(n, cu, g, seed=n, l_scale=2.0 / math.sqrt(n))
    uhf = cd > 0
    mo_dn = syn.make_system(n, cd, 1, seed=1).mo_up if uhf else None
    job = E.EngineJob(n, (cu, cd or cu), g, w, "unrestricted" if uhf else "restricted", "uhf" if uhf else "rhf", terms,
                      dt, "fp64")
    job.set_hamiltonian(0.0, sysm.h1, sysm.chol)
    job.set_trial(sysm.mo_up, mo_dn, sysm.rdm1())
    job.build_measurement()
    job.build_propagation()
    exp_h1 = np.stack([job.get(5, s).cpu().numpy() for s in range(2 if uhf else 1)])
    fields = rng.standard_normal((w, g)) + 0.3j * rng.standard_normal((w, g))
    walkers = [syn.perturbed_walkers(sysm.mo_up, w, 0.05, 1)] + ([syn.perturbed_walkers(mo_dn, w, 0.05, 2)] if uhf else [])
    dev = [torch.as_tensor(x).cuda() for x in walkers]
    f = torch.as_tensor(fields).cuda()
    names = _kernels(lambda: job.trotprop(dev[0], dev[1] if uhf else None, f))
    pick = sorted({0, min(1, w - 1), w // 2, w - 1})
    sub = [x[pick] for x in walkers]
    ref = O.apply_trotprop(sub if uhf else sub[0], fields[pick], sysm.chol, exp_h1 if uhf else exp_h1[0], dt, terms)
    for a, b in zip(dev, ref if uhf else [ref]):
        a = a.cpu().numpy()
        assert np.all(np.isfinite(a))
        assert np.max(np.abs(a[pick] - b)) < 1e-10 * np.max(np.abs(b))
    return sorted(tuple(int(x) for x in m.groups())
                  for m in (re.search(r"trot_f64_kernel<(\d+), (\d+), (\d+)>", k) for k in names) if m)


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-c{c[1]}+{c[2]}-W{c[3]}" for c in CASES])
def test_instance(case):
    print(f"[propagator tiles] {case}", flush=True)
    assert _run(*case[:4]) == [case[4]]


def test_past_the_last_size():
    print("[propagator tiles] 561", flush=True)
    assert _run(561, 9, 0, 2) == []


def test_every_instance_has_a_case():
    have = {c[4] for c in CASES}
    for mb in range(1, 5):
        for nb in range(1, 6):
            if mb * nb <= 10:
                assert {x for m, n, x in have if (m, n) == (mb, nb)} == ({0, 1, 2} if nb > 2 else {0, 1})
