"""The FP32 compensated linear stages at the edges of their tiles: 64 x 8 and
64 x 12 columns (the larger on grids with more tiles than CUs), a register
ring unrolled by 8 planes, z-chunks of any length.

One step against the FP64 oracle.  Tolerance: a stage forms differences of
values below max|q| with coefficients that sum to 284/48 per h (ACOUSTIC4)
and 612/48 per h^2 (WAVE2); with dt = 0.4 h/3, about 8 roundings on that path
and 2^-24 each, the step is within 1e-6 max|U| (ACOUSTIC4) and 1e-6 max|U|/h
(WAVE2, the second component).
"""
import numpy as np
import pytest

from test_gpu_parity import make_field, orc_grid

pytestmark = pytest.mark.gpu

CASES = [((4, 4, 4), 0), ((64, 8, 7), 0), ((65, 9, 8), 3), ((63, 12, 9), 0), ((130, 25, 17), 5), ((70, 33, 1), 0),
         ((64, 3072, 4), 0), ((60, 3061, 9), 4)]


@pytest.mark.parametrize("system,bc", [(1, (0, 0, 0)), (1, (2, 3, 0)), (1, (0, 2, 3)), (0, (0, 0, 0)), (0, (1, 0, 1))])
@pytest.mark.parametrize("n,zc", CASES, ids=[f"{n[0]}x{n[1]}x{n[2]}-zc{z}" for n, z in CASES])
def test_one_step(n, zc, system, bc, acx, orc, torch_gpu, monkeypatch):
    torch = torch_gpu
    if n[2] == 1:
        bc = (bc[0], bc[1], 0)
    if zc:
        monkeypatch.setenv("ACX_ZC_LINEAR", str(zc))
    grid = acx.Grid(n=n, h=1.0 / 64, system=system, bc=bc, c0=1.25, rho0=0.8)
    U = make_field(acx, grid, 77, "rough")
    dt = 0.4 * grid.h / 3.0 / grid.c0
    print(f"[case] linear32 n={n} zc={zc} system={system} bc={bc}", flush=True)
    ref = U.copy()
    orc.ts_solve("orc_rhs3d_cb_faithful", orc_grid(orc, grid), ref, dt, dt, 0, 4)
    st = acx.CompensatedState(grid, torch.from_numpy(U).cuda())
    st.step(dt)
    err = np.abs(st.value64().cpu().numpy() - ref).reshape(-1, grid.nvar).max(axis=0)
    scale = np.abs(U).max()
    tol = 1e-6 * scale * np.array([1.0] * 4 if system else [1.0, 1.0 / grid.h])
    print(f"[case] linear32 err {err} tol {tol}", flush=True)
    assert (err <= tol).all()
