"""Reductions at the edges of their sweeps (1024 items per block and sweep,
1024 blocks), off 16-byte alignment, and from more threads than the library
keeps scratch for.

Tolerance: sums of n positive terms by a tree of partial sums of at most 2^13
terms each differ from numpy's pairwise sum by less than 2^13 * 2^-53 = 1e-12;
maxima are exact.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [0, 1, 2, 3, 1023, 1024, 1025, 2047, 2049, 4 * 1024 * 1024 + 5]


@pytest.mark.parametrize("nvar,comp", [(1, -1), (1, 0), (3, 1), (4, -1)])
@pytest.mark.parametrize("offset", [0, 1])
def test_norms_sweep_edges(nvar, comp, offset, acx, torch_gpu):
    torch = torch_gpu
    for n in SIZES:
        X = torch.randn(n * nvar + offset, dtype=torch.float64, device="cuda",
                        generator=torch.Generator("cuda").manual_seed(n))[offset:]
        print(f"[case] norms n={n} nvar={nvar} comp={comp} offset={offset}", flush=True)
        if n == 0:
            X = torch.empty(0, dtype=torch.float64, device="cuda")
            if X.data_ptr() == 0:
                continue
        s, m = acx.norms(X, comp=comp, nvar=nvar)
        a = X.cpu().numpy()
        a = a if comp < 0 else a[comp::nvar]
        assert s == pytest.approx(float(np.sum(a * a)), rel=1e-12, abs=0.0)
        assert m == (float(np.abs(a).max()) if a.size else 0.0)


@pytest.mark.parametrize("n", [(4, 4, 4), (9, 7, 8), (33, 31, 1), (64, 65, 66)])
def test_energy_and_diff_sweep_edges(n, acx, torch_gpu):
    torch = torch_gpu
    grid = acx.Grid(n=n, h=0.1, system=acx.ACOUSTIC4, rho0=1.3, c0=0.8)
    rng = np.random.default_rng(5)
    U = rng.standard_normal(grid.shape())
    print(f"[case] energy, diff n={n}", flush=True)
    Ud = torch.from_numpy(U).cuda()
    K = 1.3 * 0.8 ** 2
    want = 0.5 * (np.sum(U[..., 0] ** 2) / K + 1.3 * np.sum(U[..., 1:] ** 2)) * 0.1 ** (2 if n[2] == 1 else 3)
    assert acx.energy(grid, Ud) == pytest.approx(want, rel=1e-12)
    hi = Ud.to(torch.float32)
    lo = (torch.randn_like(hi) * 1e-8)
    d = hi.double().cpu().numpy() + lo.double().cpu().numpy() - U
    r, m = acx.diff_f32c(hi, lo, Ud)
    assert r == pytest.approx(np.sqrt(np.sum(d * d) / np.sum(U * U)), rel=1e-12)
    assert m == np.abs(d).max()


def test_more_threads_than_scratch_slots(acx, torch_gpu):
    torch = torch_gpu
    xs = [torch.full((50000 + k,), 1.0 + k, dtype=torch.float64, device="cuda") for k in range(24)]
    torch.cuda.synchronize()
    bad = []

    def work(k):
        st = torch.cuda.Stream()
        for _ in range(20):
            s, m = acx.norms(xs[k], nvar=1, stream=st)
            if s != (50000 + k) * (1.0 + k) ** 2 or m != 1.0 + k:
                bad.append((k, s, m))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(24)]
    print("[case] norms from 24 threads", flush=True)
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad[:3]


@pytest.mark.parametrize("nvar, comp", [(1, -1), (1, 0), (3, 1), (4, -1)])
@pytest.mark.parametrize("offset", [0, 1])
def test_reductions_of_nothing(nvar, comp, offset, acx, torch_gpu):
    """No cells, with a pointer to a buffer that has some: sums and maxima of 0."""
    torch = torch_gpu
    import ctypes
    X = torch.full((64,), 7.0, dtype=torch.float64, device="cuda")[offset:]
    out = (ctypes.c_double * 2)(3.0, 3.0)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    print(f"[case] norms of no cells nvar={nvar} comp={comp} offset={offset}", flush=True)
    acx._check(acx.lib().acx_norms_f64(ptr(X), 0, nvar, comp, out, acx._stream()))
    assert tuple(out) == (0.0, 0.0)
    f = X.to(torch.float32)
    out = (ctypes.c_double * 2)(3.0, 3.0)
    acx._check(acx.lib().acx_diff_f32c_f64(ptr(f), None, ptr(X), 0, out, acx._stream()))
    assert tuple(out) == (0.0, 0.0)
