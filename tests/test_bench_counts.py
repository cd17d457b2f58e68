"""The benchmark's operation counts are those of the element kernel that runs: the marching kernel
contracts a DOF plane along x and y once for all elements that need it, so its count is well below
the per-element sum factorisation's, and a rate over that count would be no rate of the hardware."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def _march_fmas(p, mass):
    """The FP64 marching kernel's multiply-adds per lane and plane, counted loop by loop."""
    m, n = p + 1, 0
    for _ in range(m):  # U: rows
        n += 2 * m
    for _ in range(m):  # Y: Gauss points
        n += 3 * m
    for _ in range(m * m):  # Z: value (with a mass term) and gradient, and their transposes
        n += 2 * (4 if mass else 3) * m
    for _ in range(m):  # T
        n += 3 * m
    for _ in range(m):  # S
        n += 2 * m
    return n


@pytest.mark.parametrize("p", [1, 2, 3])
def test_counts_follow_the_kernel(p):
    m = p + 1
    for mass in (True, False):
        integrand = 2 * m * m if mass else 0
        assert bench.f_rhs3(p, 4, 1, False, mass) == m * (2 * _march_fmas(p, mass) + integrand)
    for variant, tiling in ((1, 1), (2, 1), (4, 0), (5, 0)):
        assert bench.f_rhs3(p, variant, tiling, False, True) == bench.f_elem(3, p)
    assert bench.f_rhs3(p, 4, 1, False, True) < 0.75 * bench.f_elem(3, p)
    assert bench.f_rhs3(p, 4, 1, True, False) < 0.75 * bench.f_elem(3, p)
    assert bench.f_march2(p, False) < 0.9 * bench.f_elem(2, p)
    assert bench.f_march2(p, False) < bench.f_march2(p, True) < bench.f_elem(2, p)
