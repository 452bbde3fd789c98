"""The z-cell 3D trace (csrc/trace3d_zcell.hip) against the oracle: grids at the
edges of its window sizes (4, 3 and 2 z-cells), uneven axes, velocity counts
that leave the last group short, one z plane, and histories whose z kicks carry
nodes out of the window, where a node forms its polynomials from the global
history and a workgroup with many of them is redone from whole slices.  rho at sampled points (exact v-sum) and the four metrics within 1e-12,
the bar of the other FP64 parity tests; rho the same bits for every launch
shape, window misses or not."""
import numpy as np
import pytest

import numericalflowiteration_amd as nufi
from numericalflowiteration_amd import config as C
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu

GRIDS = [((8, 8, 8), (6, 6, 6)), ((16, 16, 16), (7, 5, 3)), ((9, 15, 8), (8, 5, 4)), ((20, 18, 20), (6, 6, 2)),
         ((24, 24, 24), (6, 6, 2)), ((5, 4, 1), (9, 4, 5)), ((12, 3, 2), (6, 7, 3))]


def make(N, V, n):
    c = C.config_3d(N, V, 1 / 8, (n + 0.5) / 8, (0.0, 4 * np.pi), (-6.0, 6.0), C.F0_LANDAU_3D, alpha=0.05, k=0.5)
    return c


def history(c, n, strength):
    """Per slice a sum of waves, weak (one per axis) or strong (a product as well)."""
    x, y, z = (np.arange(m + 3) % m * 2 * np.pi / m for m in (c.Nx, c.Ny, c.Nz))
    out = []
    for m in range(n):
        a = 0.04 * (np.cos(x + 0.1 * m)[None, None, :] + np.cos(y)[None, :, None] + np.cos(z - 0.2 * m)[:, None, None])
        if strength == "strong":
            a = a + 4.0 * np.cos(x + 0.3 * m)[None, None, :] * np.cos(y + 0.2)[None, :, None] * np.cos(z + 0.1 * m)[:, None, None]
        out.append(a.ravel())
    return np.concatenate(out)


@pytest.mark.parametrize("strength", ["weak", "strong"])
@pytest.mark.parametrize("N,V", GRIDS)
def test_rho_and_shapes(N, V, strength):
    n = 19                                       # past the slice-15 re-wrap
    c = make(N, V, n)
    hist = history(c, n, strength)
    pts = np.unique(np.linspace(0, c.n_space() - 1, 24).astype(np.int64))
    ref = O.rho3d_points(c, n, hist, pts, exact_sum=True)
    out = []
    with nufi.GpuScheduler(c) as s:
        s.upload_history(hist, 0, n)
        for shape in [(512, 8, 1), (512, 4, 1), (256, 2, 1), (1024, 1, 1)]:
            s.set_launch_shape(*shape)
            r = np.zeros(c.n_space())
            s.compute_rho(n)
            s.download_rho(r)
            out.append(r)
        parts, cut = np.zeros(c.n_space()), c.n_nodes() // 3 + 7
        s.compute_rho(n, 0, cut)
        s.download_rho(parts)
        s.compute_rho(n, cut, c.n_nodes())
        s.download_rho(parts)
    for r in out[1:]:
        assert np.array_equal(r, out[0])
    got = out[0][pts]
    ref = ref - ref.mean() + got.mean()          # the oracle's constant ("+1") aside
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print(f"[zcell] {N} {V} {strength}: rho {err:.2e}", flush=True)
    assert err <= 1e-12
    assert np.linalg.norm(parts - out[0]) <= 1e-13 * np.linalg.norm(out[0])


@pytest.mark.parametrize("prec", [nufi.FP64, nufi.FP32C])
@pytest.mark.parametrize("strength", ["weak", "strong"])
@pytest.mark.parametrize("N,V", [((8, 8, 8), (6, 6, 6)), ((9, 7, 5), (8, 5, 4)), ((16, 16, 16), (6, 6, 2))])
def test_metrics(N, V, strength, prec):
    n = 17
    c = make(N, V, n)
    hist = history(c, n + 1, strength)
    padded = np.concatenate([hist, np.zeros(c.stride_t() + 8)])
    with nufi.GpuScheduler(c, precision=prec) as s:
        s.upload_history(hist, 0, n + 1)
        for m in (0, 1, n):
            got, parts = np.zeros(4), np.zeros(4)
            s.compute_metrics(m)
            s.download_metrics(got)
            for a, b in ((0, 11), (11, c.n_nodes())):
                s.compute_metrics(m, a, b)
                s.download_metrics(parts)
            ref = O.metrics(c, m, padded)
            assert np.max(np.abs(got - ref) / np.abs(ref)) <= 1e-12, (m, got, ref)
            assert np.max(np.abs(parts - got) / np.abs(got)) <= 1e-13
