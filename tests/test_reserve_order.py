"""Reserving a small job's block buffers: the phaseless factors are allocated before
the fields, whose capacity is what a captured block is checked against, so that a
failed allocation cannot leave room for fields without room for their factors."""
import os
import re

API = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ad_afqmc_amd", "csrc", "api.hip")


def test_factors_are_allocated_before_the_fields():
    body = re.search(r"\nint reserve_fields\(.*?\n}\n", open(API).read(), re.S).group(0)
    assert body.index("dalloc_n(&h,") < body.index("dalloc_n(&j->fields,")
    # and the capacity of each is raised only after its own allocation
    assert body.index("dalloc_n(&h,") < body.index("j->h_cap = hneed")
    assert body.index("dalloc_n(&j->fields,") < body.index("j->fields_cap = need")
