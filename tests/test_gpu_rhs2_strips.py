"""The 2D element loop in strips of 64 - p DOF columns (compute_rhs, validation.hpp:95-119) at
the edges of its split: DOF counts of one strip, one more and one fewer, few and many DOF rows,
the smallest meshes; with and without mass, reaction, k field and source. Against the oracle:
FP64 <= 1e-13 relative L2; FP32 increments of one step <= 8 u kappa^2 (u = 2^-24; the element
loop's and the solves' rounding through M^-1 of condition kappa per direction, at most 10, 30
and 90 for p = 1, 2, 3). One problem of a batch equals it run alone bit for bit."""
import numpy as np
import pytest

import adsgpu as ag
import pyoracle as po

pytestmark = pytest.mark.gpu


def _sizes(p):
    w = 64 - p  # DOF columns of a strip
    return [(w - p - 1, 7), (w - p, 1), (w - p + 1, 2), (2 * w - p + 1, 33), (1, 1), (2, 70), (p, 3 * w)]


FORMS = [dict(), dict(mass=0.0, grad=(1.0, 0.5, 0.0)), dict(reaction=1.0), dict(mass=0.0, reaction=2.0),
         dict(kfield=True), dict(kfield=True, source=True, reaction=0.5)]


@pytest.mark.parametrize("p", [1, 2, 3])
def test_strips_match_oracle(p):
    for ne in _sizes(p):
        print(f"case: strips p={p} ne={ne}", flush=True)
        g = ag.Simulation(2, [p, p], list(ne))
        o = po.Sim(2, [p, p], list(ne))
        assert g.prepare_matrices() == 0 and o.prepare_matrices() == 0
        rng = np.random.default_rng(p + sum(ne))
        c, kf, src = rng.uniform(0, 1, g.size), np.exp(rng.uniform(-0.5, 0.5, g.size)), rng.standard_normal(g.size)
        g.set(ag.U_PREV, c)
        g.set(ag.KFIELD, kf)
        g.set(ag.SOURCE, src)
        for gk in FORMS:
            g.compute_rhs(ag.rhs_form(2e-3, **gk))
            ok = dict(gk)
            if "kfield" in ok:
                ok["kfield"] = kf
            if "source" in ok:
                ok["source"] = src
            assert po.rel_l2(g.get(ag.U), o.compute_rhs(c, po.heat_form(2e-3, 2, **ok))) < 1e-13, (ne, gk)
        g.close()


@pytest.mark.parametrize("p", [1, 2, 3])
def test_fp32_increments_match_oracle(p):
    bound = 8 * 2.0**-24 * {1: 10, 2: 30, 3: 90}[p] ** 2
    for ne in _sizes(p)[:4]:
        print(f"case: strips fp32 p={p} ne={ne}", flush=True)
        g = ag.Simulation(2, [p, p], list(ne), precision=ag.FP32)
        o = po.Sim(2, [p, p], list(ne))
        assert g.prepare_matrices() == 0 and o.prepare_matrices() == 0
        u = np.random.default_rng(p + sum(ne)).uniform(0, 1, g.size)
        for gk in FORMS[:1] + FORMS[2:3]:
            g.set(ag.U, u)
            g.step(1, ag.rhs_form(1e-5, **gk))
            expect = o.solve(o.compute_rhs(u, po.heat_form(1e-5, 2, **gk))) - u
            assert po.rel_l2(g.get(ag.U) - u, expect) <= bound, (ne, gk)
        g.close()


@pytest.mark.parametrize("prec", [ag.FP64, ag.FP32])
def test_batch_of_strips_equals_single_problems(prec):
    probs = [(p, ne) for p in (1, 2, 3) for ne in (17, 64 - p, 100)]
    print(f"case: batch of strips prec={prec}", flush=True)
    form = ag.rhs_form(1e-5, reaction=1.0)
    b = ag.Batch(probs, precision=prec)
    b.prepare()
    b.set_forms([form] * len(probs))
    b.set_tuning(1, ag.TUNE_SWEEP_VARIANT)
    us = [np.random.default_rng(i).uniform(0, 1, (ne + p) ** 2) for i, (p, ne) in enumerate(probs)]
    for i, u in enumerate(us):
        b.set(i, u)
    b.step(3)
    for i, (p, ne) in enumerate(probs):
        g = ag.Simulation(2, [p, p], [ne, ne], precision=prec)
        assert g.prepare_matrices() == 0
        g.set_tuning(ag.TUNE_SWEEP_VARIANT, 1)
        g.set(ag.U, us[i])
        g.step(3, form)
        assert np.array_equal(g.get(ag.U), b.get(i)), i
        g.close()
    b.close()
