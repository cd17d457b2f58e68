"""Grids of 2^32 lanes or more wrap without an error. The segmented line sweep takes four lanes per
line of up to 16 DOFs (16 lines per wave, x lines), so on more than 2^30 such lines it leaves them to
the one-lane sweep: u = M 1, whose entries are products of the directions' basis integrals, is solved
to 1 everywhere (1e-9: the y and z lines of 32769 rows, FP64, condition of the mass matrix 10 per
direction)."""
import pytest
import torch

import adsgpu as ag

pytestmark = pytest.mark.gpu


def test_more_short_x_lines_than_segment_lanes():
    ne = (1, 32768, 32768)
    if torch.cuda.mem_get_info()[0] < 200 << 30:
        pytest.skip("needs 200 GB of device memory")
    print(f"case: ads_solve of {(ne[1] + 1) * (ne[2] + 1)} x lines", flush=True)
    g = ag.Simulation(3, [1] * 3, list(ne))
    assert g.prepare_matrices() == 0
    w = []
    for n in ne:
        a = torch.full((n + 1,), 1.0 / n, dtype=torch.float64, device="cuda")
        a[0] = a[-1] = 0.5 / n
        w.append(a)
    u = w[2][:, None, None] * w[1][None, :, None] * w[0]
    torch.cuda.synchronize()
    g.set_device(ag.U, u.data_ptr())
    g.ads_solve()
    g.get_device(ag.U, u.data_ptr())
    g.close()
    worst = max(float((plane - 1.0).abs().max()) for plane in u.split(1024))
    assert worst <= 1e-9
