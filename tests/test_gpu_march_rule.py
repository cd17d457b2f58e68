"""Which 3D element kernel a handle runs: the marching kernel (variant 4) where the mesh fills its
tiles and the device, the per-element kernels on small and thin meshes, and with a k field their
colour launches only on meshes so thin that these are faster. FP64 sums of the marching and the
per-element kernels are grouped differently, so equal bits tell that the same kernel ran."""
import numpy as np
import pytest

import adsgpu as ag
import pyoracle as po

pytestmark = pytest.mark.gpu

# default variant: step times of the marching / the best per-element kernel in us beside each
DEFAULTS = [(1, (128, 128, 128), ag.FP64, 4),  # 96 / 101
            (2, (128, 128, 128), ag.FP64, 4),  # 176 / 229
            (2, (17, 140, 140), ag.FP64, 4),  # 68 / 82
            (2, (8, 256, 256), ag.FP64, 1),  # 119 / 92
            (2, (48, 48, 48), ag.FP64, 1),  # 40 / 36
            (3, (140, 1, 140), ag.FP64, 4),  # 56 / 102
            (3, (5, 300, 300), ag.FP64, 2),  # 335 / 256
            (3, (64, 64, 64), ag.FP32, 4),  # 67 / 83
            (3, (5, 300, 300), ag.FP32, 2),  # 215 / 150
            (3, (1, 200, 200), ag.FP32, 2),  # 106 / 81
            (3, (32, 32, 32), ag.FP32, 1)]  # 42 / 37


@pytest.mark.parametrize("p,ne,precision,variant", DEFAULTS)
def test_default_variant_follows_the_mesh(p, ne, precision, variant):
    g = ag.Simulation(3, [p] * 3, list(ne), precision=precision)
    assert g.get_tuning(ag.TUNE_RHS_VARIANT) == variant
    assert g.get_tuning(ag.TUNE_RHS_TILING) == 1
    g.close()


# with a k field: does the default run the colour launches (marching / colour launches in us)
KFIELD = [(1, (5, 300, 300), True),  # 124 / 76
          (1, (24, 20, 22), False), (2, (24, 20, 22), False), (2, (5, 60, 60), False),
          (3, (3, 140, 140), True),  # 154 / 120
          (3, (18, 17, 16), False), (3, (1, 40, 40), False)]


@pytest.mark.parametrize("p,ne,colours", KFIELD)
def test_kfield_route_follows_the_mesh(p, ne, colours):
    print(f"case: k-field route p={p} ne={ne}", flush=True)
    g = ag.Simulation(3, [p] * 3, list(ne))
    o = po.Sim(3, [p] * 3, list(ne))
    rng = np.random.default_rng(p)
    u, kf = rng.uniform(0, 1, g.size), np.exp(rng.uniform(-0.5, 0.5, g.size))
    g.set(ag.U_PREV, u)
    g.set(ag.KFIELD, kf)
    out = []
    for tiling in (1, 0):
        g.set_tuning(ag.TUNE_RHS_TILING, tiling)
        g.compute_rhs(ag.rhs_form(2e-3, kfield=True))
        out.append(g.get(ag.U))
    expect = o.compute_rhs(u, po.heat_form(2e-3, 3, kfield=kf), threads=8)
    assert po.rel_l2(out[0], expect) < 1e-13 and po.rel_l2(out[1], expect) < 1e-13
    assert np.array_equal(out[0], out[1]) == colours
    g.close()
