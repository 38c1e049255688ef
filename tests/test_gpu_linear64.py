"""FP64 linear marches: linear_tile64 at the edges of its 32 x 16 tiles and
z-chunks, the marches and streaming stores for fields above the caches, and
rows of 2 GB.

Tolerance: relative L2 <= 1e-12 against the FP64 oracle, as in the parity
tests; a large grid is a small one repeated along its periodic axes, and its
result the small one's repeated.
"""
import pytest

from test_gpu_parity import TOL, make_field, orc_grid, rel_l2

pytestmark = pytest.mark.gpu

SIZES = [(32, 16, 8), (33, 17, 9), (31, 15, 7), (64, 33, 4), (5, 47, 4), (65, 4, 11), (4, 4, 4)]


@pytest.mark.parametrize("zc", [1, 3, 0])
@pytest.mark.parametrize("n", SIZES)
def test_tile_edges(n, zc, acx, orc, torch_gpu, monkeypatch):
    torch = torch_gpu
    if zc:
        monkeypatch.setenv("ACX_ZC_LINEAR", str(zc))
    for system, bcs in ((acx.ACOUSTIC4, [(0, 0, 0), (2, 3, 0), (0, 2, 3)]), (acx.WAVE2, [(0, 0, 0), (1, 0, 1)])):
        for bc in bcs:
            grid = acx.Grid(n=n, h=1.0 / 32, system=system, bc=bc, c0=1.3, rho0=0.7)
            U = make_field(acx, grid, 41, "rough")
            print(f"[case] linear64 n={n} zc={zc} system={system} bc={bc}", flush=True)
            F = orc.rhs3d(orc_grid(orc, grid), U)
            Ud = torch.from_numpy(U).cuda()
            assert rel_l2(acx.rhs(grid, Ud).cpu().numpy(), F) <= TOL
            U0 = torch.from_numpy(make_field(acx, grid, 42, "rough")).cuda()
            for a, b, c in ((0.0, 1.0, 0.01), (2.0 / 3.0, 1.0 / 3.0, 0.02)):
                out = torch.empty_like(Ud)
                acx.stage(grid, Ud, U0 if a else None, out, a, b, c)
                ref = b * U + c * F + (a * U0.cpu().numpy() if a else 0.0)
                assert rel_l2(out.cpu().numpy(), ref) <= TOL


def _repeat(t, rep):
    return t.repeat(rep[2], rep[1], rep[0], 1).contiguous()


LARGE = [((75, 45, 40), (4, 4, 4), (0, 0, 0)), ((75, 181, 40), (4, 1, 4), (0, 2, 0)),
         ((301, 45, 40), (1, 4, 4), (3, 0, 0)), ((75, 45, 163), (4, 4, 1), (0, 0, 2))]


@pytest.mark.parametrize("system", ["acoustic4", "wave2"])
@pytest.mark.parametrize("n, rep, bc", LARGE)
def test_fields_above_the_cache(n, rep, bc, system, acx, orc, torch_gpu):
    torch = torch_gpu
    kw = dict(h=1.0 / 32, system=acx.ACOUSTIC4 if system == "acoustic4" else acx.WAVE2)
    if system == "wave2":
        bc = tuple(int(k != 0) for k in bc)
    N = tuple(a * b for a, b in zip(n, rep))
    small, big = acx.Grid(n=n, bc=bc, **kw), acx.Grid(n=N, bc=bc, **kw)
    print(f"[case] large marches n={N} {system} bc={bc}", flush=True)
    U = make_field(acx, small, 43, "rough")
    F = torch.from_numpy(orc.rhs3d(orc_grid(orc, small), U)).cuda()
    U = torch.from_numpy(U).cuda()
    B, U0 = _repeat(U, rep), _repeat(torch.from_numpy(make_field(acx, small, 44, "rough")).cuda(), rep)
    assert B.numel() * 8 > 128 << 20 > U.numel() * 8
    rel = lambda x, y: float((x - y).norm() / y.norm())  # noqa: E731
    assert rel(acx.rhs(big, B), _repeat(F, rep)) <= TOL
    for a, b, c in ((0.0, 1.0, 0.01), (2.0 / 3.0, 1.0 / 3.0, 0.02)):
        out = torch.empty_like(B)
        acx.stage(big, B, U0 if a else None, out, a, b, c)
        assert rel(out, b * B + c * _repeat(F, rep) + a * U0) <= TOL


@pytest.mark.parametrize("system", ["acoustic4", "wave2"])
@pytest.mark.parametrize("n, rep, bc", [((75, 45, 40), (5, 5, 5), (0, 0, 0)), ((75, 181, 40), (5, 1, 5), (0, 2, 0))])
def test_fp32_fields_above_the_cache(n, rep, bc, system, acx, torch_gpu):
    """A compensated step of the large field against the FP64 step of the small
    one.  Tolerance as in the FP32 tile tests' derivation, for a step of 0.1 dt:
    a few roundings of 2^-24 on an increment of at most a tenth of the field."""
    torch = torch_gpu
    if system == "wave2":
        bc = tuple(int(k != 0) for k in bc)
    kw = dict(h=1.0 / 32, bc=bc, system=acx.ACOUSTIC4 if system == "acoustic4" else acx.WAVE2)
    N = tuple(a * b for a, b in zip(n, rep))
    small, big = acx.Grid(n=n, **kw), acx.Grid(n=N, **kw)
    print(f"[case] FP32 large n={N} {system} bc={bc}", flush=True)
    U = torch.from_numpy(make_field(acx, small, 46, "smooth")).cuda()
    dt = 0.1 * acx.cfl_dt(small, 0.4)
    s = acx.CompensatedState(big, _repeat(U, rep))
    assert s.hi.numel() * 4 > 80 << 20
    s.step(dt)
    ref = _repeat(acx.ssp_rks3_step(small, U.clone(), dt), rep)
    assert float((s.value64() - ref).norm() / ref.norm()) <= 1e-6


def test_rows_of_two_gigabytes(acx, torch_gpu):
    torch = torch_gpu
    m, k = 4096, 32768
    small = acx.Grid(n=(m, 4, 1), h=1.0 / 32, system=acx.WAVE2)
    big = acx.Grid(n=(m * k, 4, 1), h=1.0 / 32, system=acx.WAVE2)
    print("[case] WAVE2 rows of 2 GB", flush=True)
    U = torch.from_numpy(make_field(acx, small, 45, "rough")).cuda()
    F = acx.rhs(small, U)
    B = U.view(1, 4, 1, m, 2).expand(1, 4, k, m, 2).reshape(1, 4, m * k, 2).contiguous()
    got = acx.rhs(big, B).view(4, k, m, 2)
    ref = F.view(4, 1, m, 2)
    for j in range(0, k, 4096):   # the same arithmetic: equal to the last bit
        assert torch.equal(got[:, j:j + 4096], ref.expand(4, 4096, m, 2))


@pytest.mark.parametrize("system, rep", [("acoustic4", (3, 3, 2)), ("wave2", (3, 3, 4))])
@pytest.mark.parametrize("bc", [(0, 0, 0), (0, 0, 2)])
def test_cached_fields_on_sixteen_rows(system, rep, bc, acx, orc, torch_gpu):
    """Fields of 64 to 128 MB: 16-row tiles, cached results; the small field takes
    8-row tiles.  The same arithmetic per cell."""
    torch = torch_gpu
    kw = dict(h=1.0 / 32, system=acx.ACOUSTIC4 if system == "acoustic4" else acx.WAVE2)
    bc = tuple(int(k != 0) for k in bc) if system == "wave2" else bc
    n = (75, 45, 40) if not any(bc) else (75, 45, 40 * rep[2])
    rep = rep if not any(bc) else (rep[0], rep[1], 1)
    N = tuple(a * b for a, b in zip(n, rep))
    small, big = acx.Grid(n=n, bc=bc, **kw), acx.Grid(n=N, bc=bc, **kw)
    print(f"[case] 16-row tiles n={N} {system} bc={bc}", flush=True)
    U = make_field(acx, small, 47, "rough")
    assert rel_l2(acx.rhs(small, torch.from_numpy(U).cuda()).cpu().numpy(), orc.rhs3d(orc_grid(orc, small), U)) <= TOL
    U, U0 = torch.from_numpy(U).cuda(), torch.from_numpy(make_field(acx, small, 48, "rough")).cuda()
    B, B0 = _repeat(U, rep), _repeat(U0, rep)
    assert 64 << 20 < B.numel() * 8 <= 128 << 20 and U.numel() * 8 <= 64 << 20
    for a, b, c in ((0.0, 0.0, 1.0), (0.0, 1.0, 0.01), (2.0 / 3.0, 1.0 / 3.0, 0.02)):
        out, ref = torch.empty_like(B), torch.empty_like(U)
        acx.stage(big, B, B0 if a else None, out, a, b, c)
        acx.stage(small, U, U0 if a else None, ref, a, b, c)
        assert torch.equal(out, _repeat(ref, rep))


@pytest.mark.parametrize("nx, ny", [(1100, 4), (1100, 9), (1100, 17), (4, 1100), (17, 1100), (33, 1100)])
def test_narrow_grids_above_the_cache(nx, ny, acx, orc, torch_gpu):
    """Planes narrower than the staged region of a tile (38 x 22 cells), where
    its last rows or columns lie more than one period past the grid."""
    torch = torch_gpu
    kw = dict(h=1.0 / 32, system=acx.ACOUSTIC4)
    nz = 10
    rep = (128 << 20) // (nx * ny * nz * 32) + 1
    small, big = acx.Grid(n=(nx, ny, nz), **kw), acx.Grid(n=(nx, ny, nz * rep), **kw)
    print(f"[case] narrow march n={big.n}", flush=True)
    U = make_field(acx, small, 49, "rough")
    F = torch.from_numpy(orc.rhs3d(orc_grid(orc, small), U)).cuda()
    U = torch.from_numpy(U).cuda()
    B = _repeat(U, (1, 1, rep))
    assert B.numel() * 8 > 128 << 20
    rel = lambda x, y: float((x - y).norm() / y.norm())  # noqa: E731
    assert rel(acx.rhs(big, B), _repeat(F, (1, 1, rep))) <= TOL
    out = torch.empty_like(B)
    acx.stage(big, B, None, out, 0.0, 1.0, 0.01)
    assert rel(out, B + 0.01 * _repeat(F, (1, 1, rep))) <= TOL
