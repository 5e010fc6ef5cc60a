"""A kernel's dynamic LDS limit is state of the process, not of a launch, and jobs
may run from several host threads: it is raised in one place, once per kernel
and device and to the most that any launch takes, never to one launch's own size."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ad_afqmc_amd", "csrc")


def _sources():
    return {os.path.basename(f): open(f).read() for f in glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(
        os.path.join(CSRC, "*.h"))}


def test_limit_is_raised_in_one_place():
    calls = {f: s.count("hipFuncSetAttribute(") for f, s in _sources().items() if "hipFuncSetAttribute(" in s}
    assert calls == {"api.hip": 1}


def test_every_raise_has_a_flag_of_its_own_launcher():
    """Each call names a flag declared as a function-local static atomic just before it."""
    n = 0
    for name, s in _sources().items():
        for m in re.finditer(r"AFQ_TRY\(raise_lds\(", s):
            n += 1
            assert re.search(r"static std::atomic<uint64_t> raised\{0\};\s*(?:if \([^;{}]*\)\s*)?$", s[:m.start()]), name
    assert n >= 10
