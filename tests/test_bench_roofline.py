"""The whole-step roofline of bench.py counts the work that the engine does: the FP64
exchange contracts over the orbitals that the trial leaves empty, the reduced modes'
over all of them."""
import bench


def test_fp64_exchange_is_priced_over_the_empty_orbitals():
    N, Oa, Ob, G, m = 300, 60, 58, 2000, 10
    full, f = bench.flops_per_walker_step(N, Oa, Ob, G, m, False)
    saved = 4.0 * G * (Oa**3 + Ob**3) / m
    assert bench.whole_step_roofline(N, Oa, Ob, G, m, False, "bf16x3", 1.0)["flops_per_walker_step"] == full
    assert bench.whole_step_roofline(N, Oa, Ob, G, m, False, "fp32", 1.0)["flops_per_walker_step"] == full
    fp64 = bench.whole_step_roofline(N, Oa, Ob, G, m, False, "fp64", 1.0)
    assert abs(fp64["flops_per_walker_step"] - (full - saved)) < 1e-9 * full
    assert abs(fp64["achieved"] * 1e12 - (full - saved)) < 1e-9 * full
