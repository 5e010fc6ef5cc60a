"""Determinants, overlaps and inverses (through the Green's functions) of up to 17
electrons, where the Gauss-Jordan kernel goes from two waves to eight and a panel
is full, one short and one over, one and two spins and mixed ones, many walkers;
pivots off the diagonal; a singular matrix.  Against the oracle, 1e-10 of the
largest value, the repository's FP64 parity."""
import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn
from oracle import afqmc_oracle as O

pytestmark = pytest.mark.gpu

# (N, O up, O dn or 0, W): N past the one-work-group measurements; FP32 jobs take none of these at any N
CASES = [(160, 16, 0, 3), (200, 9, 0, 700), (200, 8, 0, 2), (300, 7, 1, 3), (200, 15, 16, 3), (160, 17, 16, 3),
         (160, 17, 1, 2)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("case", CASES + [(18, 16, 9, 5), (12, 1, 0, 4), (20, 9, 8, 3)],
                         ids=lambda c: f"N{c[0]}-O{c[1]}+{c[2]}-W{c[3]}")
def test_overlap_and_green(case, precision):
    n, ou, od, w = case
    print(f"[det/inverse small] {case} {precision}", flush=True)
    uhf = od > 0
    rng = np.random.default_rng(n + ou)
    sysm = syn.make_system(n, ou, 1, seed=n)

    def mixed(mo, seed):  # walkers mixed among their orbitals: a full overlap matrix
        o = mo.shape[1]
        u = np.linalg.qr(rng.standard_normal((o, o)) + 1j * rng.standard_normal((o, o)))[0]
        return syn.perturbed_walkers(mo, w, 0.1, seed) @ u

    mo_dn = syn.make_system(n, od, 1, seed=1).mo_up if uhf else None
    job = E.EngineJob(n, (ou, od or ou), 1, w, "unrestricted" if uhf else "restricted", "uhf" if uhf else "rhf", 2,
                      0.01, precision)
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
        assert np.max(np.abs(g.cpu().numpy().reshape(r.shape) - r)) < 1e-10 * np.max(np.abs(r))


@pytest.mark.parametrize("o", [5, 12, 16])
def test_singular_overlap(o):
    """A walker with a zero column has overlap zero; the others keep theirs."""
    n, w = 300, 4
    print(f"[det/inverse small] singular {o}", flush=True)
    sysm = syn.make_system(n, o, 1, seed=n)
    job = E.EngineJob(n, (o, o), 1, w, "restricted", "rhf", 2, 0.01, "fp32")
    job.set_hamiltonian(0.0, sysm.h1, sysm.chol)
    job.set_trial(sysm.mo_up, None, sysm.rdm1())
    job.build_measurement()
    up = syn.perturbed_walkers(sysm.mo_up, w, 0.1, 1)
    up[1, :, o - 1] = 0.0
    ov = job.overlap(torch.as_tensor(up).cuda(), None).cpu().numpy()
    ref = O.det_overlap(up, sysm.mo_up) ** 2
    assert ov[1] == 0.0
    assert np.max(np.abs(np.delete(ov, 1) - np.delete(ref, 1))) < 1e-10 * np.max(np.abs(ref))


def test_group_of_small_jobs():
    """A group none of whose jobs has more than 16 electrons a spin: one block by
    one launch per kernel against each job's own block."""
    from ad_afqmc_amd.engine import JobGroup
    from ad_afqmc_amd.serving import GpuExecutor, JobSpec

    print("[det/inverse small] group", flush=True)
    specs = [JobSpec(job_id=i, norb=n, nocc=o, nchol=g, n_walkers=w, n_steps=10, seed=20 + i, precision="bf16x3")
             for i, (n, o, g, w) in enumerate([(30, 6, 60, 33), (60, 16, 120, 17), (40, 9, 80, 20)])]
    single, grouped = (GpuExecutor(n_prop_steps=5, use_graphs=False) for _ in range(2))
    hs, hg = ([ex.start(s) for s in specs] for ex in (single, grouped))
    group = JobGroup([(h["job"], h["up"], h["weights"], h["overlaps"], h["scalars"], h["counter"], h["out"],
                       h["spec"].seed) for h in hg], 5)
    for h in hs:
        single._block(h)
    group.sr_block()
    torch.cuda.synchronize()
    for a, b in zip(hs, hg):
        for k in ("out", "weights", "overlaps", "up", "scalars"):
            x, y = b[k].cpu().numpy(), a[k].cpu().numpy()
            assert np.all(np.isfinite(x)) and np.max(np.abs(x - y)) < 1e-10 * np.max(np.abs(y))
    group.close()
    for ex, h in ((single, hs), (grouped, hg)):
        for x in h:
            ex.release(x)
