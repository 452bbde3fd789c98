"""Which kernel traces a 3D FP64 call (csrc/trace3d_zcell.hip): z-cells while the
nodes of a workgroup keep together in z, whole slices where the history drives
them apart.  Histories of each kind take the way they are meant to, the results
hold against the oracle on it (1e-12, the bar of the other FP64 parity tests), and
they depend on the history alone: the same bits after other calls, under a
replayed graph, and from the entry point that allocates nothing."""
import ctypes

import numpy as np
import pytest
import torch                  # before the library: one HIP runtime for both

import numericalflowiteration_amd as nufi
from numericalflowiteration_amd import _capi
from numericalflowiteration_amd import config as C
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu

# the window kernel's grid, a power of two in each axis, none; several passes and groups
GRIDS = [((16, 16, 16), (8, 6, 3)), ((8, 8, 8), (9, 8, 3)), ((20, 18, 12), (7, 7, 3)), ((9, 7, 10), (9, 8, 4))]
ROUTED, UNROUTED = 21, 15            # slices: decisions start at 16


def make(N, V):
    return C.config_3d(N, V, 1 / 8, 24.5 / 8, (0.0, 4 * np.pi), (-6.0, 6.0), C.F0_LANDAU_3D, alpha=0.05, k=0.5)


def history(c, n, mix):
    """Per slice one wave per axis, and `mix` times their product."""
    x, y, z = (np.arange(m + 3) % m * 2 * np.pi / m for m in (c.Nx, c.Ny, c.Nz))
    return np.concatenate([(0.04 * (np.cos(x + 0.1 * m)[None, None, :] + np.cos(y)[None, :, None] + np.cos(z - 0.2 * m)[:, None, None])
                            + mix * np.cos(x + 0.3 * m)[None, None, :] * np.cos(y + 0.2)[None, :, None] * np.cos(z + 0.1 * m)[:, None, None]).ravel()
                           for m in range(n)])


def rho_of(s, n):
    r = np.zeros(s.n_space)
    s.compute_rho(n)
    return s.download_rho(r)


def check_rho(c, n, hist, got):
    pts = np.unique(np.linspace(0, c.n_space() - 1, 20).astype(np.int64))
    ref = O.rho3d_points(c, n, hist, pts, exact_sum=True)
    ref = ref - ref.mean() + got[pts].mean()          # the oracle's constant ("+1") aside
    err = np.linalg.norm(got[pts] - ref) / np.linalg.norm(ref)
    print(f"[route] rho {err:.2e}", flush=True)
    assert err <= 1e-12


def check_metrics(c, n, hist, s):
    got = np.zeros(4)
    s.compute_metrics(n)
    s.download_metrics(got)
    ref = O.metrics(c, n, np.concatenate([hist, np.zeros(c.stride_t() + 8)]))
    assert np.max(np.abs(got - ref) / np.abs(ref)) <= 1e-12, (got, ref)


@pytest.mark.parametrize("N,V", GRIDS)
def test_separable_keeps_z_cells_and_mixing_leaves_them(N, V):
    c = make(N, V)
    for mix, window in ((0.0, False), (6.0, True)):
        hist = history(c, ROUTED + 1, mix)
        with nufi.GpuScheduler(c) as s:
            s.upload_history(hist, 0, ROUTED + 1)
            rho = rho_of(s, ROUTED)
            r = s.trace3d_route()
            print(f"[route] {N} {V} mix {mix}: {r}", flush=True)
            assert r["zcell"] and r["window"] == window
            if not window:
                assert r["spread"] < 1e-9 and r["marked"] == 0
            check_rho(c, ROUTED, hist, rho)
            check_metrics(c, ROUTED, hist, s)
            assert s.trace3d_route()["window"] == window


@pytest.mark.parametrize("N,V", GRIDS)
def test_marked_workgroups_are_redone(N, V):
    """Too few slices for a decision, and kicks that leave the window: the z-cell
    kernel reads the global history and gives up, whole slices finish."""
    c = make(N, V)
    hist = history(c, UNROUTED + 1, 12.0)
    with nufi.GpuScheduler(c) as s:
        s.upload_history(hist, 0, UNROUTED + 1)
        rho = rho_of(s, UNROUTED)
        r = s.trace3d_route()
        print(f"[route] {N} {V}: {r}", flush=True)
        assert not r["window"] and 0 < r["marked"]
        check_rho(c, UNROUTED, hist, rho)
        check_metrics(c, UNROUTED, hist, s)
        assert s.trace3d_route()["marked"] > 0


@pytest.mark.parametrize("N,V", GRIDS)
def test_bits_depend_on_the_history_alone(N, V):
    c = make(N, V)
    mixed, plain = history(c, ROUTED, 6.0), history(c, ROUTED, 0.0)
    with nufi.GpuScheduler(c) as s:
        s.upload_history(mixed, 0, ROUTED)
        first = rho_of(s, ROUTED)
        cut = c.n_nodes() // 3 + 7
        parts = np.zeros(c.n_space())
        for a, b in ((0, cut), (cut, c.n_nodes())):
            s.compute_rho(ROUTED, a, b)
            s.download_rho(parts)
        assert np.linalg.norm(parts - first) <= 1e-13 * np.linalg.norm(first)
        s.upload_history(plain, 0, ROUTED)
        unmixed = rho_of(s, ROUTED)
        rho_of(s, 5)
        s.upload_history(mixed, 0, ROUTED)
        for shape in [(512, 8, 1), (512, 4, 1), (256, 2, 1), (1024, 1, 1)]:
            s.set_launch_shape(*shape)
            assert np.array_equal(rho_of(s, ROUTED), first)
    lib, rho_dev = _capi.load(), torch.zeros(c.n_space(), dtype=torch.float64, device="cuda")
    for hist, want in ((mixed, first), (plain, unmixed), (mixed, first)):
        h = torch.tensor(np.concatenate([hist, np.zeros(8)]), dtype=torch.float64, device="cuda")
        rc = lib.nufi_rho3d_noalloc(ctypes.byref(c), ROUTED, ctypes.c_void_p(h.data_ptr()), h.numel(),
                                    ctypes.c_void_p(rho_dev.data_ptr()), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, lib.nufi_last_error(None)
        torch.cuda.synchronize()
        assert np.array_equal(rho_dev.cpu().numpy(), want)


@pytest.mark.parametrize("N,V", GRIDS[:2])
def test_replayed_graph(N, V):
    """run() over steps on both sides of the first decision, replayed with other
    work and other histories between: the bits of steps launched one by one."""
    c = make(N, V)
    first, last = 14, 20

    def steps(s, mix, graph):
        s.upload_history(history(c, first, mix), 0, first)
        s.set_run_graph(graph)
        e = s.run(first, last)
        return e, s.history(first, last)

    with nufi.GpuScheduler(c) as s:
        want = {mix: steps(s, mix, False) for mix in (6.0, 0.0)}
        for mix in (6.0, 0.0, 6.0, 0.0):
            e, h = steps(s, mix, True)
            assert np.array_equal(e, want[mix][0]) and np.array_equal(h, want[mix][1])
            rho_of(s, 3)


@pytest.mark.parametrize("N,V", [((8, 8, 8), (16, 8, 15)), ((8, 8, 8), (16, 8, 16)), ((9, 7, 10), (13, 8, 17)), ((10, 9, 8), (13, 8, 14))])
def test_metrics_on_both_sides_of_the_wave_tasks(N, V):
    """Metrics go to wave tasks below 2^20 nodes of small slices, to z-cells above."""
    c = make(N, V)
    hist = history(c, 18, 0.1)
    with nufi.GpuScheduler(c) as s:
        s.upload_history(hist, 0, 18)
        for n in (1, 17):
            check_metrics(c, n, hist, s)
        got, parts = np.zeros(4), np.zeros(4)
        s.compute_metrics(17)
        s.download_metrics(got)
        for a, b in ((0, 1000), (1000, c.n_nodes())):
            s.compute_metrics(17, a, b)
            s.download_metrics(parts)
        assert np.max(np.abs(parts - got) / np.abs(got)) <= 1e-13


@pytest.mark.parametrize("N,V", GRIDS)
def test_autotuner_has_nothing_to_choose_where_z_cells_trace(N, V):
    """Every shape would time the same launches and the pick be noise."""
    c = make(N, V)
    with nufi.GpuScheduler(c) as s:
        s.upload_history(history(c, 6, 0.0), 0, 6)
        for shape in [(1024, 1, 1), (256, 2, 1)]:
            s.set_launch_shape(*shape)
            picked, ms = s.autotune(n_probe=6, repeats=1)
            assert picked == (512, 8, 1) == s.launch_shape() and ms > 0


def test_more_than_65536_workgroups():
    """The z-cell trace takes grids of any number of workgroups, in a context and
    without allocation (a mark per workgroup in either)."""
    c = make((3, 3, 200), (6, 6, 400))
    n = 4
    hist = history(c, n, 0.1)
    with nufi.GpuScheduler(c) as s:
        s.upload_history(hist, 0, n)
        rho = rho_of(s, n)
        r = s.trace3d_route()
        print(f"[route] {r}", flush=True)
        assert r["zcell"] and r["workgroups"] > 65536
        check_rho(c, n, hist, rho)
    lib, rho_dev = _capi.load(), torch.zeros(c.n_space(), dtype=torch.float64, device="cuda")
    h = torch.tensor(np.concatenate([hist, np.zeros(8)]), dtype=torch.float64, device="cuda")
    rc = lib.nufi_rho3d_noalloc(ctypes.byref(c), n, ctypes.c_void_p(h.data_ptr()), h.numel(),
                                ctypes.c_void_p(rho_dev.data_ptr()), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.nufi_last_error(None)
    torch.cuda.synchronize()
    assert np.array_equal(rho_dev.cpu().numpy(), rho)


@pytest.mark.parametrize("N,V", [((8, 8, 8), (11, 9, 11)), ((8, 8, 8), (8, 8, 8)), ((16, 16, 16), (8, 8, 4)), ((20, 18, 20), (6, 6, 4))])
def test_first_steps(N, V):
    """rho of no, one and two slices, on both sides of the nodes at which the window
    kernel takes the first two; without allocation the same bits."""
    c = make(N, V)
    hist = history(c, 3, 0.1)
    lib, rho_dev = _capi.load(), torch.zeros(c.n_space(), dtype=torch.float64, device="cuda")
    h = torch.tensor(np.concatenate([hist, np.zeros(8)]), dtype=torch.float64, device="cuda")
    with nufi.GpuScheduler(c) as s:
        s.upload_history(hist, 0, 3)
        for n in (0, 1, 2):
            rho = rho_of(s, n)
            check_rho(c, n, hist, rho)
            rc = lib.nufi_rho3d_noalloc(ctypes.byref(c), n, ctypes.c_void_p(h.data_ptr()), h.numel(),
                                        ctypes.c_void_p(rho_dev.data_ptr()), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
            assert rc == 0, lib.nufi_last_error(None)
            torch.cuda.synchronize()
            assert np.array_equal(rho_dev.cpu().numpy(), rho)
