"""The device adjoint where its layout changes: rings shorter than a wave and
barely longer than a cell's four points, node counts that leave the last
workgroup short, 256-, 512- and 1024-thread workgroups, several chunks of
slices, and grids too wide for per-cell adjoints (folded ones instead).  The
gradient against the oracle's forward tangent at the bars of the other adjoint
tests: 1e-8 of its largest entry in FP64, 1e-5 in FP32C."""
import numpy as np
import pytest

import numericalflowiteration_amd as nufi
from numericalflowiteration_amd import adjoint as A
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(nufi.FP64, 1e-8), (nufi.FP32C, 1e-5)])
@pytest.mark.parametrize("Nx,Nu,T", [(5, 33, 1.0), (64, 200, 4.5), (100, 96, 2.5), (48, 2000, 0.5), (64, 4500, 0.25),
                                     (2048, 16, 0.5), (3000, 12, 0.5)])
def test_gradient(Nx, Nu, T, prec, tol):
    conf = nufi.multimode_1d(nufi.adjoint_modes(), Nx=Nx, Nu=Nu, T=T)
    J, g = A.energy_and_grad(conf, nufi.adjoint_modes(), precision=prec)
    Jt, dJ = O.tangent_run(conf)
    err = np.max(np.abs(g - dJ[:8])) / np.max(np.abs(dJ[:8]))
    print(f"[adjoint {Nx} x {Nu}] precision={prec} J rel err {abs(J - Jt) / abs(Jt):.3e}, grad vs tangent {err:.3e}", flush=True)
    assert err <= tol
