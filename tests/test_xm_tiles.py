"""The tiles of the 1D x-major launches (trace1d_xm_setup, make_tile,
make_xm_node, xm_reduce of csrc/trace1d.hip): the same integer arithmetic on
the CPU (every node of a range traced by one thread, every LDS slot and partial
written once), and on the GPU rho of uneven grids and ranges against the oracle
(exact v-sum, the 1e-12 and 1e-6 bars of the other parity tests)."""
import math

import numpy as np
import pytest

import numericalflowiteration_amd as nufi
from numericalflowiteration_amd import config as C
from tests import oracle_lib as O

GROUP, CUS = 16, 256


def tile(ix_count, Nu, block, npt, spread):
    ppx = -(-Nu // GROUP)
    k0, k1 = -(-ix_count // 64), -(-ix_count // 16)
    if spread:
        k = min(max(CUS // ppx, k0), k1)
        xw, rows = -(-ix_count // k), GROUP
    else:
        unit, best, xw, rows = GROUP // min(GROUP, npt), 0, 0, 0
        for c in range(k0, k1 + 1):
            w = -(-ix_count // c)
            r = block // w // unit * unit
            used = ix_count * r * 65536 // c
            if r > 0 and used > best:
                best, xw, rows = used, w, r
    n_xt = -(-ix_count // xw)
    return xw, rows, n_xt, -(-xw * rows // 64) * 64


@pytest.mark.parametrize("block,npt,spread", [(1024, 1, True), (1024, 1, False), (512, 2, False), (256, 4, False),
                                              (512, 4, False), (1024, 2, False)])
@pytest.mark.parametrize("ix_count,Nu", [(1, 16), (7, 33), (25, 40), (64, 17), (100, 35), (129, 48), (256, 20)])
def test_every_node_has_one_thread(ix_count, Nu, block, npt, spread):
    xw, rows, n_xt, threads = tile(ix_count, Nu, block, npt, spread)
    assert 0 < xw <= 64 and rows > 0 and (rows * npt) % GROUP == 0
    assert xw * rows <= threads <= block
    if spread:
        assert xw <= 64 and (n_xt * -(-Nu // GROUP) <= CUS or xw > 32 or n_xt == -(-ix_count // 64))
    traced = np.zeros((ix_count, Nu), dtype=int)
    written = np.zeros((ix_count, -(-Nu // GROUP)), dtype=int)
    for wg in range(n_xt * -(-Nu // (rows * npt))):
        xt, vb = wg % n_xt, wg // n_xt
        slot = np.zeros(rows * npt * xw, dtype=int)
        for t in range(threads):
            vr = t // xw
            xo = t - vr * xw
            for r in range(npt):
                vi = r * rows + vr
                if vr < rows:
                    slot[vi * xw + xo] += 1
                    ix, iu = xt * xw + xo, vb * npt * rows + vi
                    if ix < ix_count and iu < Nu:
                        traced[ix, iu] += 1
        assert (slot == 1).all() and slot.size <= block * npt
        for k in range(rows * npt // GROUP * xw):
            xl, gg = xt * xw + k % xw, vb * (rows * npt // GROUP) + k // xw
            if xl < ix_count and gg < written.shape[1]:
                written[xl, gg] += 1
    assert (traced == 1).all() and (written == 1).all()


@pytest.mark.gpu
@pytest.mark.parametrize("prec,tol", [(nufi.FP64, 1e-12), (nufi.FP32C, 1e-6)])
@pytest.mark.parametrize("Nx,Nu", [(7, 33), (17, 16), (25, 100), (64, 256), (100, 515), (129, 48), (256, 40)])
def test_rho_of_uneven_grids(Nx, Nu, prec, tol):
    conf = C.config_1d(Nx, Nu, 1 / 16, 3.0, 0.0, 4 * math.pi, -10.0, 10.0, C.F0_LANDAU_1D, 0.05, 0.5)
    n, st = 40, conf.stride_t()
    j = np.arange(st) % Nx
    hist = np.concatenate([0.03 * np.cos(2 * np.pi * j / Nx + 0.2 * m) for m in range(n)])
    N, cut = conf.n_nodes(), Nu * (Nx // 3) + 5
    with nufi.GpuScheduler(conf, precision=prec) as s:
        s.upload_history(hist, 0, n)
        whole, parts = np.zeros(Nx), np.zeros(Nx)
        s.compute_rho(n)
        s.download_rho(whole)
        for a, b in ((0, cut), (cut, N)):               # two ranges of other tiles
            s.compute_rho(n, a, b)
            s.download_rho(parts)
    exact = O.rho(conf, n, hist, exact_sum=True) - 1.0
    for r in (whole, parts):
        err = np.linalg.norm((r - r.mean()) - (exact - exact.mean())) / np.linalg.norm(exact - exact.mean())
        assert err <= tol, err
