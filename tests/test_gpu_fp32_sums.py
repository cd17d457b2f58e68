"""FP32 element loops (compute_rhs, validation.hpp:95-119): the sums of different elements are FP64
and the derivatives come from differences inside an element, so the right-hand side is no further
from FP64 than per-element FP32 contributions summed in FP64.

The bars compare errors of two FP32 evaluations of the same entries against the FP64 oracle: each
rounds the same contractions in another order, so their root-mean-square errors over a whole mesh
and three states are alike; 1.1 leaves room for the spread. The second evaluation is that of the
per-element kernels in 3D and the per-element loop in numpy's float32 in 2D. Sums of the elements
in FP32 are beyond the bar (1.2 to 1.4 with a k field in 3D, 1.13 to 1.18 in 2D)."""
import numpy as np
import pytest

import adsgpu as ag
import pyoracle as po

pytestmark = pytest.mark.gpu

DT = 2.0**-14


def _f32(x):
    return np.asarray(x, dtype=np.float32).astype(np.float64)


def _increment(g, u, form):
    """The FP32 handle's rhs - M u_prev."""
    g.set(ag.U, u)
    g.swap()
    g.compute_rhs(form)
    return g.get(ag.BUFFER)


@pytest.mark.parametrize("p,ne", [(1, (20, 18, 16)), (2, (20, 21, 19)), (3, (18, 17, 20)), (3, (33, 30, 36))])
def test_march_error_is_no_larger_than_per_element_kernels(p, ne):
    print(f"case: fp32 sums 3D p={p} ne={ne}", flush=True)
    g = ag.Simulation(3, [p] * 3, list(ne), precision=ag.FP32)
    o = po.Sim(3, [p] * 3, list(ne))
    assert g.prepare_matrices() == 0 and o.prepare_matrices() == 0
    kf = _f32(np.exp(0.4 * np.sin(np.arange(g.size) * 0.01)))
    g.set(ag.KFIELD, kf)
    forms = [dict(), dict(reaction=1.0, grad=(0.0625, 0.0625, 0.125))]
    if p < 3:  # at p = 3 a k field stays on the per-element kernels
        forms.append(dict(kfield=True))
    for gk in forms:
        ok = dict(gk, kfield=kf) if gk.get("kfield") else gk
        err = {1: 0.0, 4: 0.0}
        for seed in range(3):
            u = _f32(o.init_gaussians(seed=seed, count=4, sigma=(0.05, 0.15), centre=(0.2, 0.8), noise=1e-3))
            expect = o.compute_rhs(u, po.heat_form(DT, 3, mass=0.0, **ok))
            for variant in err:
                g.set_tuning(ag.TUNE_RHS_VARIANT, variant)
                # (in one launch a k field always marches)
                g.set_tuning(ag.TUNE_RHS_TILING, 1 if variant == 4 else 0)
                err[variant] += po.rel_l2(_increment(g, u, ag.rhs_form(DT, **gk)), expect) ** 2
        assert err[4] <= 1.1**2 * err[1], (gk, err)
    g.close()


@pytest.mark.parametrize("p", [1, 2, 3])
def test_a_spike_leaves_other_elements_alone(p):
    """A line of coefficients of 1e6 along z, in the middle of the tiles along x: the rhs of DOFs
    whose elements do not hold them is that of the state without it."""
    mid = {1: 15, 2: 9, 3: 8}[p]
    ne = (2 * mid + 8, 9, 13)
    print(f"case: fp32 spike p={p} ne={ne}", flush=True)
    g = ag.Simulation(3, [p] * 3, list(ne), precision=ag.FP32)
    o = po.Sim(3, [p] * 3, list(ne))
    assert g.prepare_matrices() == 0 and o.prepare_matrices() == 0
    u = _f32(o.init_gaussians(seed=2, count=4, sigma=(0.05, 0.15), centre=(0.2, 0.8), noise=1e-3))
    shape = [n + p for n in ne][::-1]
    spiked = u.copy().reshape(shape)
    spiked[:, ::4, mid] = 1e6
    spiked = spiked.ravel()
    away = np.abs(np.arange(shape[2]) - mid) > p  # x beyond every element that holds the spike
    out = []
    for variant, state in ((1, u), (4, u), (4, spiked)):
        g.set_tuning(ag.TUNE_RHS_VARIANT, variant)
        out.append(_increment(g, state, ag.rhs_form(DT)).reshape(shape)[:, :, away])
    expect = o.compute_rhs(u, po.heat_form(DT, 3, mass=0.0)).reshape(shape)[:, :, away]
    assert po.rel_l2(out[1], expect) <= 1.1 * po.rel_l2(out[0], expect)
    assert np.array_equal(out[2], out[1])
    g.close()


def _per_element(o, p, ne, u, mass, grad):
    """mass u v - dt grad u . grad v: every element's contributions in float32, summed in FP64."""
    t = [o.tables(d) for d in (0, 1)]
    (bx, dx, wx), (by, dy, wy) = [[np.float32(a) for a in (d["b"][:, :, 0], d["b"][:, :, 1], d["J"][:, None] * d["w"])]
                                  for d in t]
    m, shape = p + 1, (ne[1] + p, ne[0] + p)
    ey, ex = np.arange(ne[1]), np.arange(ne[0])
    iy, ix = ey[:, None] + np.arange(m), ex[:, None] + np.arange(m)
    c = np.float32(u.reshape(shape))[iy[:, None, :, None], ix[None, :, None, :]]  # [ey][ex][b][a]

    def dot(spec, a, b):  # one index, its products added one by one
        return np.einsum(spec, a, b, optimize=False).astype(np.float32)
    a0, a1 = dot("yxba,xqa->yxbq", c, bx), dot("yxba,xqa->yxbq", c, dx)
    v, vx, vy = (dot("yxbq,yrb->yxrq", s, t) for s, t in ((a0, by), (a1, by), (a0, dy)))
    w = wy[:, None, :, None] * wx[None, :, None, :]
    k = np.float32(-DT * grad) * w
    g0, gx, gy = np.float32(mass) * w * v, k * vx, k * vy
    h = dot("yxrq,yrb->yxbq", g0, by) + dot("yxrq,yrb->yxbq", gy, dy)
    hx = dot("yxrq,yrb->yxbq", gx, by)
    r = dot("yxbq,xqa->yxba", h, bx) + dot("yxbq,xqa->yxba", hx, dx)
    out = np.zeros(shape)
    np.add.at(out, (np.broadcast_to(iy[:, None, :, None], r.shape), np.broadcast_to(ix[None, :, None, :], r.shape)),
              r.astype(np.float64))
    return _f32(out).ravel()


@pytest.mark.parametrize("p,ne", [(1, (40, 33)), (2, (77, 60)), (3, (64, 64)), (3, (228, 190))])
def test_strip_error_is_that_of_element_contributions_summed_in_fp64(p, ne):
    print(f"case: fp32 sums 2D p={p} ne={ne}", flush=True)
    g = ag.Simulation(2, [p, p], list(ne), precision=ag.FP32)
    o = po.Sim(2, [p, p], list(ne))
    assert g.prepare_matrices() == 0 and o.prepare_matrices() == 0
    for mass, grad in ((0.0, 1.0), (1.0, 0.0)):
        gpu = emulated = 0.0
        for seed in range(3):
            u = _f32(np.random.default_rng(seed).uniform(0, 1, g.size))
            # an FP32 handle's form has its mass term reduced by 1
            got = _increment(g, u, ag.rhs_form(DT, mass=1.0 + mass, grad=(grad,) * 3))
            expect = o.compute_rhs(u, po.heat_form(DT, 2, mass=mass, grad=(grad,) * 3))
            gpu += po.rel_l2(got, expect) ** 2
            emulated += po.rel_l2(_per_element(o, p, ne, u, mass, grad), expect) ** 2
        assert gpu <= 1.1**2 * emulated, (mass, grad, gpu**0.5, emulated**0.5)
    g.close()
