"""adsg_autotune in 2D: the element loop is one kernel whatever the element variant and the tiling,
and the tiling chooses the k-field gradient's kernels (one launch for the adjoint pair, or colour
launches), which a timed step does not run. So the autotuner leaves both as the handle has them,
also when the choices come from the cache, and picks the line sweep only."""
import numpy as np
import pytest

import adsgpu as ag

pytestmark = pytest.mark.gpu

ELEMENT_KEYS = (ag.TUNE_RHS_VARIANT, ag.TUNE_RHS_COLUMNS, ag.TUNE_RHS_TILING)


@pytest.mark.parametrize("cache", [0, 1])
@pytest.mark.parametrize("dim_config", [dict(), dict(quad_order=[4, 4])])
def test_autotune_keeps_the_element_settings(cache, dim_config):
    print(f"case: autotune 2D cache={cache} {dim_config}", flush=True)
    handles = []
    for tiling, variant in ((1, 2), (0, 3), (1, 0)):
        if dim_config and tiling:
            continue  # general configurations have no one-launch tiling
        g = ag.Simulation(2, [2, 2], [61, 47], **dim_config)
        g.prepare_matrices()
        g.set(ag.U, np.random.default_rng(1).uniform(0, 1, g.size))
        g.set(ag.KFIELD, np.ones(g.size))
        g.set_tuning(ag.TUNE_CACHE, cache)
        g.set_tuning(ag.TUNE_RHS_TILING, tiling)
        g.set_tuning(ag.TUNE_RHS_VARIANT, variant)
        before = [g.get_tuning(k) for k in ELEMENT_KEYS]
        u = g.get(ag.U)
        g.autotune(ag.rhs_form(1e-6, kfield=True))
        assert [g.get_tuning(k) for k in ELEMENT_KEYS] == before
        assert g.get_tuning(ag.TUNE_SWEEP_VARIANT) in (0, 1, 2)
        assert np.array_equal(g.get(ag.U), u)
        handles.append(g)
    for g in handles:
        g.close()
