"""The FP64 nonlinear stage kernel at the edges of its tiles: output tiles are
30 x 10 (ACOUSTIC4) and 30 x 14 (WAVE2) columns, z-chunks end anywhere.

Each case prints its name before the GPU call.  Tolerance: relative L2 <=
1e-12 against the FP64 oracle (about 300 operations per value on O(1) data at
2^-53, with the 4th power of the indicators and a margin of 10).
"""
import numpy as np
import pytest

from test_gpu_parity import TOL, make_field, orc_grid, rel_l2

pytestmark = pytest.mark.gpu

SIZES = [(30, 10, 8), (31, 11, 7), (29, 9, 13), (60, 14, 4), (61, 15, 5), (4, 29, 6)]


@pytest.mark.parametrize("zc", [1, 3, 0])
@pytest.mark.parametrize("n", SIZES)
def test_tile_edges(n, zc, acx, orc, torch_gpu, monkeypatch):
    torch = torch_gpu
    if zc:
        monkeypatch.setenv("ACX_ZC_CWENO", str(zc))
    for system, bcs in ((acx.ACOUSTIC4, [(0, 0, 0), (2, 3, 0), (0, 2, 3)]), (acx.WAVE2, [(0, 0, 0), (1, 0, 1)])):
        for bc in bcs:
            grid = acx.Grid(n=n, h=1.0 / n[1], system=system, bc=bc, gamma_hi=0.85, gamma_lo=0.85, c0=1.3, rho0=0.7)
            U = make_field(acx, grid, 31, "step")
            print(f"[case] cweno64 n={n} zc={zc} system={system} bc={bc}", flush=True)
            g = orc_grid(orc, grid)
            F = orc.rhs3d(g, U)
            Ud = torch.from_numpy(U).cuda()
            assert rel_l2(acx.rhs(grid, Ud).cpu().numpy(), F) <= TOL
            # the stage epilogues: a*U0 + b*Q + c*F(Q)
            U0 = torch.from_numpy(make_field(acx, grid, 32, "rough")).cuda()
            for a, b, c in ((0.0, 1.0, 0.01), (2.0 / 3.0, 1.0 / 3.0, 0.02)):
                out = torch.empty_like(Ud)
                acx.stage(grid, Ud, U0 if a else None, out, a, b, c)
                ref = b * U + c * F + (a * U0.cpu().numpy() if a else 0.0)
                assert rel_l2(out.cpu().numpy(), ref) <= TOL
