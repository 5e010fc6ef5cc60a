"""Overlaps and Green's functions around the sizes where the Gauss-Jordan kernel
changes (65, 128, 129 electrons) and at the edges of its panels and of the rows
a lane holds, one and two spins, against the oracle: 1e-10 of the largest value,
the repository's FP64 parity."""
import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, O up, O dn or 0, W): permute the rows of the walkers so that pivots move
CASES = [(70, 65, 0, 3), (90, 66, 79, 2), (96, 80, 64, 2), (100, 81, 7, 3), (120, 96, 97, 2), (140, 112, 113, 2),
         (140, 127, 0, 5), (150, 128, 1, 2), (150, 129, 128, 2)]


@pytest.mark.parametrize("case", CASES, ids=[f"N{c[0]}-O{c[1]}+{c[2]}" for c in CASES])
def test_overlap_and_green(case):
    n, ou, od, w = case
    print(f"[det/inverse] {case}", flush=True)
    uhf = od > 0
    rng = np.random.default_rng(n + ou)
    sysm = syn.make_system(n, ou, 1, seed=n)
    # trial orbitals in scrambled order and walkers mixed among themselves: the
    # overlap matrix is a full one whose pivots are off the diagonal
    def mixed(mo, seed):
        o = mo.shape[1]
        u = np.linalg.qr(rng.standard_normal((o, o)) + 1j * rng.standard_normal((o, o)))[0]
        return syn.perturbed_walkers(mo, w, 0.1, seed) @ u
    mo_dn = syn.make_system(n, od, 1, seed=1).mo_up if uhf else None
    job = E.EngineJob(n, (ou, od or ou), 1, w, "unrestricted" if uhf else "restricted", "uhf" if uhf else "rhf", 2,
                      0.01, "fp64")
    job.set_hamiltonian(0.0, sysm.h1, sysm.chol)
    job.set_trial(sysm.mo_up, mo_dn, sysm.rdm1())
    job.build_measurement()
    walkers = [mixed(sysm.mo_up, 1)] + ([mixed(mo_dn, 2)] if uhf else [])
    dev = [torch.as_tensor(x).cuda() for x in walkers]
    ov = job.overlap(dev[0], dev[1] if uhf else None).cpu().numpy()
    ref = O.det_overlap(walkers[0], sysm.mo_up)
    ref = ref * O.det_overlap(walkers[1], mo_dn) if uhf else ref ** 2
    assert np.max(np.abs(ov - ref) / np.abs(ref)) < 1e-10
    got = job.green(dev[0], dev[1] if uhf else None)
    got = list(got) if isinstance(got, (tuple, list)) else [got]
    for g, x, mo in zip(got, walkers, [sysm.mo_up, mo_dn]):
        r = O.green(x, mo)
        g = g.cpu().numpy().reshape(r.shape)
        assert np.max(np.abs(g - r)) < 1e-10 * np.max(np.abs(r))
