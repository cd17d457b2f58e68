"""The segmented line sweeps (dgbtrs on every line, band_solve.hpp:20-31) at the edges of
their split: the shortest segmented line, lines of exactly 16 k rows and one more or fewer,
the longest lines whose x staging fits the LDS in FP64 and the first ones whose staging does
not, the change to segments of 32 rows, and line counts of one wave and one more. Plain and
transposed solves against the oracle.

FP64 <= 1e-13 relative L2. FP32 handles solve inside their increment steps: the increment of
one step from random coefficients, whose right-hand side and backward stable band solves each
give 4 u kappa^2 (u = 2^-24, kappa the condition of a direction's mass matrix, at most 10, 30
and 90 for p = 1, 2, 3 with the open knot vector's end rows)."""
import numpy as np
import pytest

import adsgpu as ag
import pyoracle as po

pytestmark = pytest.mark.gpu

# line lengths in x against y
SIZES = [(17, 64), (18, 65), (32, 17), (33, 31), (48, 63), (49, 48), (193, 20), (208, 33), (209, 17), (224, 18),
         (225, 19), (256, 66), (257, 17), (288, 20)]


def _pair(p, nx, ny, precision):
    print(f"case: segment edges p={p} n={nx}x{ny} prec={precision}", flush=True)
    g = ag.Simulation(2, [p, p], [nx - p, ny - p], precision=precision)
    o = po.Sim(2, [p, p], [nx - p, ny - p])
    assert g.prepare_matrices() == 0 and o.prepare_matrices() == 0
    return g, o


@pytest.mark.parametrize("p", [1, 2, 3])
def test_solves_at_segment_edges_match_oracle(p):
    for nx, ny in SIZES:
        g, o = _pair(p, nx, ny, ag.FP64)
        b = np.random.default_rng(nx + p).standard_normal(g.size)
        for transposed in (False, True):
            g.set(ag.U, b)
            if transposed:
                g.ads_solve_transposed()
            else:
                g.ads_solve()
            expect = o.solve(b.copy(), transposed=transposed)
            assert po.rel_l2(g.get(ag.U), expect) <= 1e-13, (nx, ny, transposed)
        g.close()


@pytest.mark.parametrize("p", [1, 2, 3])
def test_fp32_increments_at_segment_edges_match_oracle(p):
    dt, bound = 1e-5, 8 * 2.0**-24 * {1: 10, 2: 30, 3: 90}[p] ** 2
    for nx, ny in SIZES:
        g, o = _pair(p, nx, ny, ag.FP32)
        u = np.random.default_rng(nx + p).standard_normal(g.size)
        g.set(ag.U, u)
        g.step(1, ag.rhs_form(dt))
        r = o.compute_rhs(u, po.heat_form(dt, 2))
        assert po.rel_l2(g.get(ag.U) - u, o.solve(r) - u) <= bound, (nx, ny)
        g.close()


@pytest.mark.parametrize("p", [1, 2, 3])
def test_one_segment_lines_match_oracle_and_transposed_stays_refused(p):
    """Lines of at most 16 DOFs: one segment, the plain solve only."""
    for nx, ny in [(p + 1, p + 1), (p + 2, 16), (15, 17), (16, 40), (16, p + 1)]:
        g, o = _pair(p, nx, ny, ag.FP64)
        b = np.random.default_rng(nx + ny + p).standard_normal(g.size)
        g.set(ag.U, b)
        g.ads_solve()
        assert po.rel_l2(g.get(ag.U), o.solve(b.copy())) <= 1e-13, (nx, ny)
        with pytest.raises(ag.AdsgError):
            g.ads_solve_transposed()
        g.close()
