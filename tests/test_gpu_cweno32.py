"""FP32 CWENO stages where flagged and unflagged cells share wavefronts, at the
edges of the 30 x 14 x 8 patch tiles.

One selective step with a flagged slab: away from its border (four stages of 3
cells) the flagged part equals the FP64 CWENO step, the rest the FP64 linear
step.  Tolerance: a face value carries a few FP32 roundings, at most 4 x 2^-24
of the field, and enters the step with a weight of at most dt c / h = 0.4:
relative L2 <= 1e-7.  Non-finite data beside an unflagged cell's arms (in the
corner and diagonal slots only the nonlinear weights read) leaves it finite.
"""
import numpy as np
import pytest

from test_gpu_parity import make_field, rel_l2

pytestmark = pytest.mark.gpu


def _step64(acx, torch, n, gamma, bc, U, dt):
    g = acx.Grid(n=n, h=1.0 / 96, bc=bc, gamma_hi=gamma[0], gamma_lo=gamma[1])
    return acx.ssp_rks3_step(g, U.clone(), dt).cpu().numpy()


@pytest.mark.parametrize("bc", [(0, 0, 0), (0, 3, 0)])
@pytest.mark.parametrize("n", [(96, 14, 8), (93, 15, 9), (90, 29, 17), (96, 13, 7)])
def test_slab_of_flags(n, bc, acx, torch_gpu):
    torch = torch_gpu
    grid = acx.Grid(n=n, h=1.0 / 96, bc=bc, gamma_hi=0.85, gamma_lo=0.85)
    U = torch.from_numpy(make_field(acx, grid, 7, "step")).cuda()
    dt = acx.cfl_dt(grid, 0.4)
    fl = torch.zeros((n[2], n[1], n[0]), dtype=torch.uint8, device="cuda")
    fl[:, :, :48] = 15
    print(f"[case] flagged slab n={n} bc={bc}", flush=True)
    s = acx.CompensatedState(grid, U)
    s.step(dt, flags=fl.reshape(-1))
    got = s.value64().cpu().numpy()
    cw = _step64(acx, torch, n, (0.85, 0.85), bc, U, dt)
    lin = _step64(acx, torch, n, (1.0, 0.0), bc, U, dt)
    assert rel_l2(got[:, :, 12:36], cw[:, :, 12:36]) <= 1e-7
    assert rel_l2(got[:, :, 60:76], lin[:, :, 60:76]) <= 1e-7
    if rel_l2(lin[:, :, 12:36], cw[:, :, 12:36]) > 1e-6:   # the schemes differ there
        assert rel_l2(got[:, :, 12:36], lin[:, :, 12:36]) > 5e-7


@pytest.fixture
def clean(acx, torch_gpu):
    """No non-finite report of this test is left to the next."""
    acx.nonfinite_clear()
    yield
    torch_gpu.cuda.synchronize()
    acx.nonfinite_clear()


def test_unflagged_component_ignores_diagonal_neighbours(acx, torch_gpu, clean):
    torch = torch_gpu
    n = (32, 16, 8)
    grid = acx.Grid(n=n, h=1.0 / 32, gamma_hi=0.85, gamma_lo=0.85)
    U = torch.from_numpy(make_field(acx, grid, 9, "smooth")).cuda()
    U[4, 8, 16, 0] = float("nan")
    fl = torch.zeros((n[2], n[1], n[0]), dtype=torch.uint8, device="cuda")
    fl[2, 2, 2] = 15   # marks the tile; its cells' arms do not reach the NaN
    print("[case] NaN on a diagonal of unflagged cells", flush=True)
    s = acx.CompensatedState(grid, U)
    s.step(1e-4, flags=fl.reshape(-1))
    got = s.value64().cpu().numpy()
    bad = ~np.isfinite(got).all(-1)
    # four stages spread the NaN along the axes, 3 cells a stage and axis
    z, y, x = np.nonzero(bad)
    dist = np.abs(x - 16) + np.abs(y - 8) + np.minimum(np.abs(z - 4), 8 - np.abs(z - 4))
    assert bad.any() and dist.max() <= 12


@pytest.mark.parametrize("bc", [(0, 0, 0), (0, 3, 0)])
@pytest.mark.parametrize("n", [(96, 14, 8), (93, 15, 9), (90, 29, 17), (96, 13, 7)])
def test_flagged_slab_is_not_the_linear_scheme(n, bc, acx, torch_gpu):
    """A jump inside the compared part of the flagged slab and one inside the
    unflagged part: the schemes differ there by far more than either tolerance,
    and each part takes its own."""
    torch = torch_gpu
    grid = acx.Grid(n=n, h=1.0 / 96, bc=bc, gamma_hi=0.85, gamma_lo=0.85)
    rng = np.random.default_rng(8)
    x = np.arange(n[0])[None, None, :, None]
    U = np.where((x // 24) % 2 == 0, 1.0, 0.1) + 0.01 * rng.standard_normal(grid.shape())
    U = torch.from_numpy(U).cuda()
    dt = acx.cfl_dt(grid, 0.4)
    fl = torch.zeros((n[2], n[1], n[0]), dtype=torch.uint8, device="cuda")
    fl[:, :, :48] = 15
    print(f"[case] jumps in and out of the flagged slab n={n} bc={bc}", flush=True)
    s = acx.CompensatedState(grid, U)
    s.step(dt, flags=fl.reshape(-1))
    got = s.value64().cpu().numpy()
    cw = _step64(acx, torch, n, (0.85, 0.85), bc, U, dt)
    lin = _step64(acx, torch, n, (1.0, 0.0), bc, U, dt)
    for part, want, other in ((slice(12, 36), cw, lin), (slice(60, 76), lin, cw)):
        assert rel_l2(other[:, :, part], want[:, :, part]) > 1e-4
        assert rel_l2(got[:, :, part], want[:, :, part]) <= 1e-7
        assert rel_l2(got[:, :, part], other[:, :, part]) > 1e-5
