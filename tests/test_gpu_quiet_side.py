"""The nonlinear reconstruction beside a jump, cell by cell on the smooth side.

One half of the grid holds a small background, the other a field of order one.
The smooth sided stencil of a background cell at the jump takes all the weight
(the others: (background^2 / jump^2)^4, below 1e-40), so its face states, and
with them the right-hand side of the background cells behind it, carry the
rounding of the background, not that of the jump.  Errors are maxima over those
cells, relative to their largest right-hand side or increment.

FP64: TOL, 1e-12 (about 300 operations of 2^-53, margin 10), against the FP64
oracle.  FP32: face states of some 16 roundings of 2^-24 of the background, a
difference of two in a right-hand side: 4e-6.  The step of the FP32 test is so
short (dt c / h = 1e-6) that what later stages bring in from the jump, of the
order of dt^2, is exact to far less than that.
"""
import numpy as np
import pytest

from test_gpu_parity import TOL, make_field, orc_grid

pytestmark = pytest.mark.gpu

N = (36, 34, 32)
AXES = {"x": 2, "y": 1, "z": 0}


def jump_field(grid, axis, jump, background, seed):
    """(field, mask of the background cells that are not next to the jump)."""
    rng = np.random.default_rng(seed)
    shape = grid.shape()
    n = shape[AXES[axis]]
    at = np.arange(n).reshape([-1 if d == AXES[axis] else 1 for d in range(3)])
    quiet = np.broadcast_to(at < n // 2, shape[:3])
    U = np.where(quiet[..., None], background, jump) * (1.0 + 0.3 * rng.standard_normal(shape))
    return U, np.broadcast_to((at >= 1) & (at < n // 2 - 1), shape[:3])


@pytest.mark.parametrize("axis", AXES)
@pytest.mark.parametrize("system", ["acoustic4", "wave2"])
@pytest.mark.parametrize("jump, background", [(1.0, 1e-8), (1e3, 1e-6), (1e-2, 1e-12)])
def test_fp64_rhs_behind_a_jump(jump, background, system, axis, acx, orc, torch_gpu):
    torch = torch_gpu
    grid = acx.Grid(n=N, h=1.0 / 32, system=acx.ACOUSTIC4 if system == "acoustic4" else acx.WAVE2,
                    gamma_hi=0.85, gamma_lo=0.85)
    U, quiet = jump_field(grid, axis, jump, background, 5)
    print(f"[case] quiet side FP64 {system} {axis} jump {jump:g} background {background:g}", flush=True)
    F = orc.rhs3d(orc_grid(orc, grid), U)[quiet]
    got = acx.rhs(grid, torch.from_numpy(U).cuda()).cpu().numpy()[quiet]
    assert np.abs(F).max() < 1e3 * background * 32 * 32
    err = np.abs(got - F).max(0) / np.abs(F).max(0)
    print(f"[case] largest error {err.max():.1e}", flush=True)
    assert (err <= TOL).all()


@pytest.mark.parametrize("axis", AXES)
@pytest.mark.parametrize("jump, background", [(1.0, 1e-5), (1e3, 1e-3)])
@pytest.mark.parametrize("flagged", [False, True])
def test_fp32_step_behind_a_jump(flagged, jump, background, axis, acx, torch_gpu):
    torch = torch_gpu
    grid = acx.Grid(n=N, h=1.0 / 32, gamma_hi=0.85, gamma_lo=0.85)
    U, quiet = jump_field(grid, axis, jump, background, 6)
    U = torch.from_numpy(U.astype(np.float32).astype(np.float64)).cuda()
    dt = 1e-6 * grid.h
    print(f"[case] quiet side FP32 {axis} jump {jump:g} background {background:g} flagged {flagged}", flush=True)
    s = acx.CompensatedState(grid, U)
    s.step(dt, flags=torch.full((grid.ncells,), 15, dtype=torch.uint8, device="cuda") if flagged else None)
    ref = (acx.ssp_rks3_step(grid, U.clone(), dt) - U).cpu().numpy()[quiet]
    got = (s.value64() - U).cpu().numpy()[quiet]
    err = np.abs(got - ref).max(0) / np.abs(ref).max(0)
    print(f"[case] largest error {err.max():.1e}", flush=True)
    assert (err <= 4e-6).all()


def test_fp32_indicators_of_large_fields(acx, torch_gpu):
    """A field of 2e18, whose indicators are below the largest FP32 number, takes
    the step of the field of order one, times its size, to the rounding of the
    faces (relative L2 <= 1e-7, as for the flagged slabs of the FP32 stages)."""
    torch = torch_gpu
    grid = acx.Grid(n=(32, 28, 24), h=1.0 / 32, gamma_hi=0.85, gamma_lo=0.85)
    U = torch.from_numpy(make_field(acx, grid, 31, "step") / 1.75).cuda()
    amp = 2e18
    print(f"[case] FP32 nonlinear weights of fields of {amp:g}", flush=True)
    acx.nonfinite_clear()
    try:
        got = []
        for a in (1.0, amp):
            s = acx.CompensatedState(grid, U * a)
            s.step(acx.cfl_dt(grid, 0.4))
            got.append(s.value64() / a)
        assert float((got[1] - got[0]).norm() / got[0].norm()) <= 1e-7
    finally:
        torch.cuda.synchronize()
        acx.nonfinite_clear()
