"""3D slices whose pads are not the periodic copies of their interior: a trace
reads the pads as they stand, as the reference does (fields.hpp:308-350), on every
path, from uploaded histories, after steps, and in the entry point that allocates
nothing.  Against the oracle, which reads them too, at the 1e-12 of the other FP64
parity tests."""
import ctypes

import numpy as np
import pytest
import torch                  # before the library: one HIP runtime for both

import numericalflowiteration_amd as nufi
from numericalflowiteration_amd import _capi
from numericalflowiteration_amd import config as C
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu

GRIDS = [((16, 16, 16), (6, 6, 4)), ((8, 8, 8), (9, 8, 3)), ((9, 7, 10), (9, 8, 4)), ((5, 4, 2), (9, 4, 5))]


def make(N, V):
    return C.config_3d(N, V, 1 / 8, 24.5 / 8, (0.0, 4 * np.pi), (-6.0, 6.0), C.F0_LANDAU_3D, alpha=0.05, k=0.5)


def history(c, n, axis, odd):
    """n slices of one wave per axis; in those with odd(m) the pads of `axis` (0 x, 1 y, 2 z) are another wave's."""
    x, y, z = (np.arange(m + 3) % m * 2 * np.pi / m for m in (c.Nx, c.Ny, c.Nz))
    out = []
    for m in range(n):
        a = 0.04 * (np.cos(x + 0.1 * m)[None, None, :] + np.cos(y)[None, :, None] + np.cos(z - 0.2 * m)[:, None, None])
        if odd(m):
            N = (c.Nx, c.Ny, c.Nz)[axis]
            at = [slice(None)] * 3
            at[2 - axis] = slice(N, N + 3)
            a[tuple(at)] += 0.03 * np.sin(1.0 + np.arange(a[tuple(at)].size)).reshape(a[tuple(at)].shape)
        out.append(a.ravel())
    return np.concatenate(out)


def check_rho(c, n, hist, got):
    pts = np.arange(c.n_space()) if c.n_space() < 100 else np.unique(np.r_[np.linspace(0, c.n_space() - 1, 16).astype(np.int64),
                                                                          c.n_space() - 1, c.Nx - 1, c.Nx * c.Ny - 1])
    ref = O.rho3d_points(c, n, hist, pts, exact_sum=True)
    ref = ref - ref.mean() + got[pts].mean()          # the oracle's constant ("+1") aside
    err = np.linalg.norm(got[pts] - ref) / np.linalg.norm(ref)
    print(f"[pads] rho {err:.2e}", flush=True)
    assert err <= 1e-12


def check(c, n, hist, s):
    rho = np.zeros(c.n_space())
    s.compute_rho(n)
    s.download_rho(rho)
    check_rho(c, n, hist, rho)
    got = np.zeros(4)
    s.compute_metrics(n)
    s.download_metrics(got)
    ref = O.metrics(c, n, np.concatenate([hist, np.zeros(c.stride_t() + 8)]))
    assert np.max(np.abs(got - ref) / np.abs(ref)) <= 1e-12, (got, ref)


@pytest.mark.parametrize("n", [4, 20])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("N,V", GRIDS)
def test_pads_are_read_as_they_stand(N, V, axis, n):
    c = make(N, V)
    hist = history(c, n + 1, axis, lambda m: m in (1, n - 1))
    with nufi.GpuScheduler(c) as s:
        s.upload_history(hist, 0, n + 1)
        check(c, n, hist, s)
        plain = history(c, n + 1, axis, lambda m: False)
        s.upload_history(plain, 0, n + 1)                 # and periodic ones again
        check(c, n, plain, s)
    lib, rho_dev = _capi.load(), torch.zeros(c.n_space(), dtype=torch.float64, device="cuda")
    h = torch.tensor(np.concatenate([hist, np.zeros(8)]), dtype=torch.float64, device="cuda")
    rc = lib.nufi_rho3d_noalloc(ctypes.byref(c), n, ctypes.c_void_p(h.data_ptr()), h.numel(),
                                ctypes.c_void_p(rho_dev.data_ptr()), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.nufi_last_error(None)
    torch.cuda.synchronize()
    check_rho(c, n, hist, rho_dev.cpu().numpy())


@pytest.mark.parametrize("N,V", GRIDS[:2])
def test_steps_after_odd_slices(N, V):
    """run() from odd slices, by a graph captured before them, and over them."""
    c = make(N, V)
    first, last = 3, 6
    plain, odd = history(c, first, 0, lambda m: False), history(c, first, 0, lambda m: m == 1)
    with nufi.GpuScheduler(c) as s:
        s.upload_history(plain, 0, first)
        e0 = s.run(first, last)
        s.upload_history(odd, 0, first)
        e1 = s.run(first, last)
        h1 = s.history(0, last)
        rho = np.zeros(c.n_space())
        s.compute_rho(last)
        s.download_rho(rho)
        check_rho(c, last, h1, rho)
        s.upload_history(odd, 0, first)
        s.set_run_graph(False)
        assert np.array_equal(e1, s.run(first, last)) and not np.array_equal(e0, e1)
        s.set_run_graph(True)
        s.run(0, last)                                    # overwrites the odd slice
        s.upload_history(plain, 0, first)
        assert np.array_equal(e0, s.run(first, last))
