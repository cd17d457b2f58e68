"""The one-launch tiling's spill fix-up on meshes with many short rows of DOFs along x, which take
a lane per DOF (rows of fewer than 56 DOFs, 8192 of them or more): against the colour launches, whose
sums are grouped differently (1e-14, as for the other meshes), with fixed boundaries against the
oracle's step (1e-12, as for other steps), and on a mesh with more rows than one wave per row can
be launched for (2^26), where the rhs of u = 1 is the product of the directions' basis integrals."""
import numpy as np
import pytest

import adsgpu as ag
import pyoracle as po

pytestmark = pytest.mark.gpu

# rows at the edges of the rule: 8190 (lane per DOF not taken), 8192, more; 55 and 56 DOFs
MESHES = [(1, (1, 89, 90)), (1, (1, 127, 63)), (2, (5, 126, 62)), (3, (2, 90, 95)), (1, (54, 95, 92)), (2, (54, 95, 92))]


@pytest.mark.parametrize("p,ne", MESHES)
def test_short_rows_match_colours_and_oracle(p, ne):
    print(f"case: fix-up of short rows p={p} ne={ne}", flush=True)
    for variant in (1, 4):
        g = ag.Simulation(3, [p] * 3, list(ne))
        g.set_tuning(ag.TUNE_RHS_VARIANT, variant)
        g.set(ag.U_PREV, np.random.default_rng(p).uniform(0, 1, g.size))
        out = []
        for tiling in (0, 1, 1):
            g.set_tuning(ag.TUNE_RHS_TILING, tiling)
            g.compute_rhs(ag.rhs_form(2e-3, reaction=1.0))
            out.append(g.get(ag.U))
        assert po.rel_l2(out[1], out[0]) < 1e-14
        assert np.array_equal(out[1], out[2])
        g.close()
    g = ag.Simulation(3, [p] * 3, list(ne))
    o = po.Sim(3, [p] * 3, list(ne))
    g.fix_all_boundaries()
    o.fix_all_boundaries()
    assert g.prepare_matrices() == 0 and o.prepare_matrices() == 0
    u = np.random.default_rng(p).uniform(0, 1, g.size)
    o.zero_boundary(u)
    g.set(ag.U, u)
    g.step(1, ag.rhs_form(1e-6), ag.STEP_DIRICHLET)
    rhs = o.compute_rhs(u, po.heat_form(1e-6, 3), threads=8)
    o.zero_boundary(rhs)
    expect = o.solve(rhs)
    assert po.rel_l2(g.get(ag.U), expect) <= 1e-12
    g.close()


def test_more_rows_than_a_wave_each():
    ne = (1, 8192, 8192)
    print(f"case: fix-up of 2^26 rows ne={ne}", flush=True)
    g = ag.Simulation(3, [1] * 3, list(ne))
    g.set(ag.U_PREV, np.ones(g.size))
    g.compute_rhs(ag.rhs_form(1.0))
    got = g.get(ag.U).reshape([n + 1 for n in ne][::-1])
    g.close()
    w = [np.full(n + 1, 1.0 / n) for n in ne]  # integrals of the hat functions
    for a in w:
        a[0] = a[-1] = 0.5 * a[0]
    got /= w[2][:, None, None] * w[1][None, :, None] * w[0]
    # (u = 1 has no gradient up to rounding: differences of 1 against 1, of 8192 eps each)
    assert np.abs(got - 1.0).max() <= 8 * 8192**2 * 2.0**-52
