"""The marching element kernel (variant 4 in one launch, and every k-field form in one launch)
at the edges of its tiles: 31 / 19 / 16 elements along x for p = 1 / 2 / 3, 4 along y, and along
z the chunk that rhs3_march_tiles chooses (4 on these meshes, so counts of 4 n and 4 n +- 1),
against the oracle's element loop. FP64 bar: the sums of at most (2p + 2)^3 rounded products per
entry in another order, 1e-13 as for the other one-launch kernels; FP32: the 1e-6 of FP32 steps."""
import numpy as np
import pytest

import adsgpu as ag
import pyoracle as po

pytestmark = pytest.mark.gpu

MESHES = [(1, (31, 4, 8)), (1, (32, 5, 9)), (1, (30, 3, 3)), (1, (63, 9, 1)),
          (2, (19, 8, 12)), (2, (20, 5, 13)), (2, (18, 3, 11)), (2, (39, 2, 4)), (2, (1, 9, 5)),
          (3, (16, 4, 16)), (3, (17, 5, 15)), (3, (15, 7, 9)), (3, (33, 1, 6)), (3, (2, 6, 17))]


def _pair(p, ne, precision=ag.FP64, dirichlet=False):
    g = ag.Simulation(3, [p] * 3, list(ne), precision=precision)
    o = po.Sim(3, [p] * 3, list(ne))
    if dirichlet:
        g.fix_all_boundaries()
        o.fix_all_boundaries()
    assert g.prepare_matrices() == 0 and o.prepare_matrices() == 0
    g.set_tuning(ag.TUNE_RHS_VARIANT, 4)
    g.set_tuning(ag.TUNE_RHS_TILING, 1)
    return g, o


@pytest.mark.parametrize("p,ne", MESHES)
def test_march_rhs_matches_oracle(p, ne):
    print(f"case: march rhs p={p} ne={ne}", flush=True)
    g, o = _pair(p, ne)
    rng = np.random.default_rng(61 + p)
    c, kf, src = rng.uniform(0, 1, g.size), np.exp(rng.uniform(-0.5, 0.5, g.size)), rng.standard_normal(g.size)
    g.set(ag.U_PREV, c)
    g.set(ag.KFIELD, kf)
    g.set(ag.SOURCE, src)
    dt = 2e-3
    for gk in (dict(), dict(mass=0.0, grad=(1.0, 0.5, 2.0)), dict(reaction=1.0), dict(kfield=True),
               dict(kfield=True, mass=0.0, grad=(0.5, 2.0, 1.0)), dict(kfield=True, reaction=0.5),
               dict(source=True), dict(kfield=True, source=True, reaction=0.5)):
        ok = {k: v for k, v in gk.items() if k not in ("kfield", "source")}
        if gk.get("kfield"):
            ok["kfield"] = kf
        if gk.get("source"):
            ok["source"] = src
        expect = o.compute_rhs(c, po.heat_form(dt, 3, **ok))
        g.compute_rhs(ag.rhs_form(dt, **gk))
        first = g.get(ag.U)
        assert po.rel_l2(first, expect) < 1e-13, gk
        g.compute_rhs(ag.rhs_form(dt, **gk))  # the start value is written, not added to
        assert np.array_equal(g.get(ag.U), first), gk
    g.close()


@pytest.mark.parametrize("p,ne", [(1, (32, 5, 9)), (2, (20, 5, 13)), (2, (39, 2, 4)), (3, (17, 5, 15))])
def test_march_fp32_steps_and_delta_steps_match_oracle(p, ne):
    """FP32 increments against the FP64 oracle's steps, with a constant far larger than the
    variation of the state (the kernel takes a constant out of the gradient forms), with fixed
    rows, a k field (per-element kernels at p = 3) and, as delta steps, a source."""
    print(f"case: march fp32 p={p} ne={ne}", flush=True)
    dt = 1e-5
    for dirichlet, kfield in ((False, False), (True, False), (False, True)):
        g, o = _pair(p, ne, ag.FP32, dirichlet)
        u = o.init_gaussians(seed=31, count=3, sigma=(0.05, 0.15), centre=(0.2, 0.8), noise=1e-3)
        if dirichlet:
            o.zero_boundary(u)
        else:
            u = u + 50.0
        kf = np.exp(np.random.default_rng(3).uniform(-0.5, 0.5, g.size))
        g.set(ag.U, u)
        g.set(ag.KFIELD, kf)
        for _ in range(3):
            rhs = o.compute_rhs(u, po.heat_form(dt, 3, kfield=kf) if kfield else po.heat_form(dt, 3))
            if dirichlet:
                o.zero_boundary(rhs)
            u = o.solve(rhs)
            g.step(1, ag.rhs_form(dt, kfield=kfield), ag.STEP_DIRICHLET if dirichlet else 0)
            assert po.rel_l2(g.get(ag.U), u) <= 1e-6
        g.close()
    for precision, tol in ((ag.FP64, 1e-12), (ag.FP32, 1e-6)):
        g, o = _pair(p, ne, precision)
        u = o.init_gaussians(seed=7, count=3, sigma=(0.05, 0.15), centre=(0.2, 0.8), noise=1e-3)
        src = np.random.default_rng(4).standard_normal(g.size)
        g.set(ag.U, u)
        g.set(ag.SOURCE, src)
        f = po.heat_form(dt, 3, source=src)
        f.mass = 0.0
        for _ in range(2):
            u = u + o.solve(o.compute_rhs(u, f))
            g.step_delta(1, ag.rhs_form(dt, mass=0.0, source=True), [0, 0, 0])
            assert po.rel_l2(g.get(ag.U), u) <= tol
        g.close()
