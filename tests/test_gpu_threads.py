"""Distinct jobs of different sizes, each from a host thread and on a stream of its
own at once: steps and energies bit for bit those of the same calls one job after
another.  The jobs share kernels whose dynamic LDS differs by size."""
import math
import threading

import numpy as np
import pytest
import torch

from ad_afqmc_amd import engine as E
from ad_afqmc_amd import synthetic as syn

pytestmark = pytest.mark.gpu

# (N, O, G, W): one work-group a walker, few occupied with other LDS needs, wide
SIZES = [(16, 4, 30, 40), (46, 15, 90, 20), (100, 20, 60, 33), (130, 70, 20, 6)]


def _job(n, o, g, w):
    s = syn.make_system(n, o, g, seed=n, l_scale=2.0 / math.sqrt(n))
    job = E.EngineJob(n, (o, o), g, w, "restricted", "rhf", 6, 0.01, "fp64")
    job.set_hamiltonian(0.0, s.h1, s.chol)
    job.set_trial(s.mo_up, None, s.rdm1())
    job.build_measurement()
    job.build_propagation()
    up = torch.as_tensor(syn.perturbed_walkers(s.mo_up, w, 0.05, 1)).cuda()
    fields = torch.as_tensor(np.random.default_rng(n).standard_normal((6, w, g))).cuda()
    return job, up, fields


def _run(job, up, fields, out):
    with torch.cuda.stream(torch.cuda.Stream()):
        x = up.clone()
        weights = torch.ones(x.shape[0], dtype=torch.float64, device="cuda")
        overlaps = job.overlap(x, None)
        scalars = torch.tensor([-1.0, -1.0], dtype=torch.float64, device="cuda")
        for f in fields:
            job.propagate(x, None, f, weights, overlaps, scalars, None)
            out.append(job.energy(x, None))
        out += [x, weights, overlaps]
        torch.cuda.current_stream().synchronize()


def test_concurrent_jobs_equal_serial_ones():
    print("[threads]", flush=True)
    jobs = [_job(*c) for c in SIZES]
    torch.cuda.synchronize()
    serial = [[] for _ in jobs]
    for j, o in zip(jobs, serial):
        _run(*j, o)
    for _ in range(5):
        outs, errors = [[] for _ in jobs], []

        def call(j, o):
            try:
                _run(*j, o)
            except Exception as e:  # noqa: BLE001
                errors.append(e)

        threads = [threading.Thread(target=call, args=(j, o)) for j, o in zip(jobs, outs)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors
        for a, b in zip(outs, serial):
            assert len(a) == len(b) and all(torch.equal(x, y) for x, y in zip(a, b))
