"""Rules by the size of a call: 3D metrics of slabs (wave tasks) and of whole grids
(z-cells) add up and hold against the oracle, 1D tiles with a narrower last one, partial
sums of one lane a point past 64 and its multiples, and transforms of lines without
small factors, in four terms at a time and the rest; 3D rho of the first steps.  The 1e-12 (FP64) and 1e-6 (FP32C)
of the other parity tests."""
import ctypes

import numpy as np
import pytest
import torch                  # before the library: one HIP runtime for both

import numericalflowiteration_amd as nufi
from numericalflowiteration_amd import _capi
from numericalflowiteration_amd import config as C
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu


def wave3(c, n):
    x, y, z = (np.arange(m + 3) % m * 2 * np.pi / m for m in (c.Nx, c.Ny, c.Nz))
    return np.concatenate([0.04 * (np.cos(x + 0.1 * m)[None, None, :] + np.cos(y)[None, :, None] + np.cos(z - 0.2 * m)[:, None, None]).ravel()
                           for m in range(n)])


@pytest.mark.parametrize("N,V", [((16, 16, 16), (8, 6, 3)), ((20, 18, 12), (7, 7, 3)), ((8, 8, 8), (16, 8, 18)), ((13, 12, 9), (9, 8, 13))])
def test_metrics_of_slabs_add_up(N, V):
    c = C.config_3d(N, V, 1 / 8, 24.5 / 8, (0.0, 4 * np.pi), (-6.0, 6.0), C.F0_LANDAU_3D, alpha=0.05, k=0.5)
    n, total = 17, c.n_nodes()
    hist = wave3(c, n + 1)
    with nufi.GpuScheduler(c) as s:
        s.upload_history(hist, 0, n + 1)
        whole = np.zeros(4)
        s.compute_metrics(n)
        s.download_metrics(whole)
        for pieces in (2, 7, 29):
            cuts, parts = np.linspace(0, total, pieces + 1).astype(np.int64), np.zeros(4)
            for a, b in zip(cuts[:-1], cuts[1:]):
                s.compute_metrics(n, int(a), int(b))
                s.download_metrics(parts)
            assert np.max(np.abs(parts - whole) / np.abs(whole)) <= 1e-13, pieces
    ref = O.metrics(c, n, np.concatenate([hist, np.zeros(c.stride_t() + 8)]))
    assert np.max(np.abs(whole - ref) / np.abs(ref)) <= 1e-12


# one lane a point with 64, 65, 130 partials; tables past 16 KiB; 64-wide tiles and 2, 1, 22 points more
@pytest.mark.parametrize("prec,tol", [(nufi.FP64, 1e-12), (nufi.FP32C, 1e-6)])
@pytest.mark.parametrize("Nx,Nu", [(130, 1400), (257, 1024), (300, 1040), (65, 4100), (150, 2080), (700, 60), (1500, 33)])
def test_rho_tiles_and_partials(Nx, Nu, prec, tol):
    c = C.config_1d(Nx, Nu, 1 / 16, 1.5, 0.0, 4 * np.pi, -10.0, 10.0, C.F0_LANDAU_1D, 0.05, 0.5)
    n, st = 18, c.stride_t()
    j = np.arange(st) % Nx
    hist = np.concatenate([0.03 * np.cos(2 * np.pi * j / Nx + 0.2 * m) for m in range(n)])
    cut = Nu * (Nx // 3) + 5
    with nufi.GpuScheduler(c, precision=prec) as s:
        s.upload_history(hist, 0, n)
        whole, parts = np.zeros(Nx), np.zeros(Nx)
        s.compute_rho(n)
        s.download_rho(whole)
        for a, b in ((0, cut), (cut, c.n_nodes())):
            s.compute_rho(n, a, b)
            s.download_rho(parts)
    exact = O.rho(c, n, hist, exact_sum=True) - 1.0
    for r in (whole, parts):
        err = np.linalg.norm((r - r.mean()) - (exact - exact.mean())) / np.linalg.norm(exact - exact.mean())
        print(f"[sizes] {Nx} x {Nu} {prec}: {err:.2e}", flush=True)
        assert err <= tol


@pytest.mark.parametrize("prec", [nufi.FP64, nufi.FP32C])
@pytest.mark.parametrize("Nx", [5, 6, 7, 11, 13, 22, 33, 97, 102, 721])
def test_lines_without_small_factors(Nx, prec):
    """Nodal values through the spline fit and back (FP32C contexts: the direct transform)."""
    c = C.config_1d(Nx, 16, 1 / 16, 0.5, 0.0, 4 * np.pi, -10.0, 10.0, C.F0_LANDAU_1D, 0.05, 0.5)
    v = np.cos(0.37 * np.arange(Nx)) + 0.2 * np.sin(1.1 * np.arange(Nx) + 0.5)
    with nufi.GpuScheduler(c, precision=prec) as s:
        a = np.asarray(s.interpolate(v)).ravel()[:Nx + 3]
    back = (a[:Nx] + 4 * a[1:Nx + 1] + a[2:Nx + 2]) / 6
    assert np.linalg.norm(back - v) <= 1e-12 * np.linalg.norm(v)
    assert np.array_equal(a[Nx:], a[:3])


@pytest.mark.parametrize("N,V", [((32, 8, 8), (64, 8, 2)), ((16, 8, 8), (20, 16, 5)), ((10, 9, 10), (16, 16, 9)), ((20, 20, 20), (8, 8, 2)),
                                 ((12, 12, 12), (8, 8, 6))])
def test_first_steps_3d(N, V):
    """rho of up to four slices by whichever kernel; without allocation the same bits."""
    c = C.config_3d(N, V, 1 / 8, 24.5 / 8, (0.0, 4 * np.pi), (-6.0, 6.0), C.F0_LANDAU_3D, alpha=0.05, k=0.5)
    hist = wave3(c, 4)
    pts = np.unique(np.linspace(0, c.n_space() - 1, 12).astype(np.int64))
    lib, rho_dev = _capi.load(), torch.zeros(c.n_space(), dtype=torch.float64, device="cuda")
    h = torch.tensor(np.concatenate([hist, np.zeros(8)]), dtype=torch.float64, device="cuda")
    with nufi.GpuScheduler(c) as s:
        s.upload_history(hist, 0, 4)
        for n in (1, 2, 3, 4):
            rho = np.zeros(c.n_space())
            s.compute_rho(n)
            s.download_rho(rho)
            ref = O.rho3d_points(c, n, hist, pts, exact_sum=True)
            ref = ref - ref.mean() + rho[pts].mean()          # the oracle's constant ("+1") aside
            assert np.linalg.norm(rho[pts] - ref) <= 1e-12 * np.linalg.norm(ref)
            rc = lib.nufi_rho3d_noalloc(ctypes.byref(c), n, ctypes.c_void_p(h.data_ptr()), h.numel(),
                                        ctypes.c_void_p(rho_dev.data_ptr()), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
            assert rc == 0, lib.nufi_last_error(None)
            torch.cuda.synchronize()
            assert np.array_equal(rho_dev.cpu().numpy(), rho)
