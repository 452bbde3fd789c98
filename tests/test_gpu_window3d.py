"""The 3D FP64 window kernel and the wave-task metrics (csrc/trace3d.hip) on grids
of fewer than 32 (u, v) velocities, which no z-cell plan takes: every workgroup
size and node count, chunks of several slices, one and two LDS buffers, re-wraps at
slices 15 and 31, and ranges cut inside a point.  Against the oracle at the 1e-12
of the other FP64 parity tests; the same bits for every launch shape."""
import numpy as np
import pytest

import numericalflowiteration_amd as nufi
from numericalflowiteration_amd import config as C
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu

# 16^3 (compiled strides), a power of two, uneven axes, slices too wide for two buffers
GRIDS = [((16, 16, 16), (5, 5, 3)), ((8, 8, 8), (5, 6, 4)), ((9, 7, 5), (5, 5, 5)), ((20, 19, 18), (4, 5, 2))]
SHAPES = [(512, 8, 1), (512, 4, 1), (512, 2, 1), (512, 1, 1), (256, 8, 1), (256, 4, 1), (256, 2, 1), (256, 1, 1), (1024, 8, 1),
          (1024, 4, 1), (1024, 2, 1), (1024, 1, 1), (512, 4, 2), (256, 2, 3), (1024, 1, 5)]
N_STEP = 35


def make(N, V):
    return C.config_3d(N, V, 1 / 8, (N_STEP + 0.5) / 8, (0.0, 4 * np.pi), (-6.0, 6.0), C.F0_LANDAU_3D, alpha=0.05, k=0.5)


def history(c, n, mix):
    x, y, z = (np.arange(m + 3) % m * 2 * np.pi / m for m in (c.Nx, c.Ny, c.Nz))
    return np.concatenate([(0.04 * (np.cos(x + 0.1 * m)[None, None, :] + np.cos(y)[None, :, None] + np.cos(z - 0.2 * m)[:, None, None])
                            + mix * np.cos(x + 0.3 * m)[None, None, :] * np.cos(y + 0.2)[None, :, None] * np.cos(z + 0.1 * m)[:, None, None]).ravel()
                           for m in range(n)])


@pytest.mark.parametrize("mix", [0.0, 0.5])
@pytest.mark.parametrize("N,V", GRIDS)
def test_rho_and_shapes(N, V, mix):
    c = make(N, V)
    hist = history(c, N_STEP, mix)
    pts = np.unique(np.linspace(0, c.n_space() - 1, 20).astype(np.int64))
    ref = O.rho3d_points(c, N_STEP, hist, pts, exact_sum=True)
    with nufi.GpuScheduler(c) as s:
        assert not s.trace3d_route()["zcell"]
        s.upload_history(hist, 0, N_STEP)
        out = []
        for shape in SHAPES:
            try:
                s.set_launch_shape(*shape)
            except nufi.NufiError:
                assert shape[2] > 1, shape                 # several wide slices do not fit the LDS
                continue
            r = np.zeros(c.n_space())
            s.compute_rho(N_STEP)
            s.download_rho(r)
            out.append((shape, r))
        parts, cut = np.zeros(c.n_space()), c.n_nodes() // 3 + 7
        for a, b in ((0, cut), (cut, c.n_nodes())):
            s.compute_rho(N_STEP, a, b)
            s.download_rho(parts)
    assert len(out) >= 12
    rho = out[0][1]
    for shape, r in out[1:]:
        assert np.array_equal(r, rho), shape
    ref = ref - ref.mean() + rho[pts].mean()               # the oracle's constant ("+1") aside
    err = np.linalg.norm(rho[pts] - ref) / np.linalg.norm(ref)
    print(f"[window] {N} {V} mix {mix}: rho {err:.2e}, {len(out)} shapes", flush=True)
    assert err <= 1e-12
    assert np.linalg.norm(parts - rho) <= 1e-13 * np.linalg.norm(rho)


@pytest.mark.parametrize("mix", [0.0, 0.5])
@pytest.mark.parametrize("N,V", GRIDS)
def test_metrics(N, V, mix):
    c = make(N, V)
    hist = history(c, 19, mix)
    with nufi.GpuScheduler(c) as s:
        s.upload_history(hist, 0, 19)
        for n in (0, 1, 18):
            got, parts = np.zeros(4), np.zeros(4)
            s.compute_metrics(n)
            s.download_metrics(got)
            for a, b in ((0, 11), (11, c.n_nodes())):
                s.compute_metrics(n, a, b)
                s.download_metrics(parts)
            ref = O.metrics(c, n, np.concatenate([hist, np.zeros(c.stride_t() + 8)]))
            assert np.max(np.abs(got - ref) / np.abs(ref)) <= 1e-12, (n, got, ref)
            assert np.max(np.abs(parts - got) / np.abs(got)) <= 1e-13
