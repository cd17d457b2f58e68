"""FP32 element loops (compute_rhs, validation.hpp:95-119): the sums of different elements are FP64
and the derivatives come from differences inside an element, so the right-hand side is no further
from FP64 than per-element FP32 contributions summed in FP64.

The bars compare errors of two FP32 evaluations of the same entries against the FP64 oracle: each
rounds the same contractions in another order, so their root-mean-square errors over a whole mesh
and three states are alike; 1.1 leaves room for the spread. The second evaluation is that of the
per-element kernels on the same input. Sums of the elements in FP32 are beyond the bar (1.2 to 1.4
with a k field)."""
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
