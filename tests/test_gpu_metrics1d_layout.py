"""1D metrics where the kernel's layout changes: node counts that leave the last
wave and workgroup short, 256-, 512- and 1024-thread workgroups, field grids off
the powers of two, tables that take one LDS buffer or (widest) do not fit it at
all, metrics grids beyond the field grid's period, and cuts of the node range.
Against the oracle at the 1e-12 of the other metrics tests."""
import numpy as np
import pytest

import numericalflowiteration_amd as nufi
from numericalflowiteration_amd import config as C
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu


def landau(Nx, Nu, x0=0.0):
    return C.config_1d(Nx, Nu, 1 / 16, 1.5, x0, x0 + 4 * np.pi, -8.0, 8.0, C.F0_LANDAU_1D, alpha=0.05, k=0.5)


@pytest.mark.parametrize("field,nodes,x0", [((16, 40), (5, 33), 0.0), ((32, 64), (100, 700), 0.0), ((30, 64), (64, 1100), 0.0),
                                            ((64, 64), (128, 2100), 0.0), ((49, 64), (48, 64), 9.0), ((64, 64), (31, 65), -20.0),
                                            ((4000, 8), (40, 50), 0.0), ((8000, 8), (40, 50), 0.0)])
def test_metrics(field, nodes, x0):
    conf, cm = landau(*field), landau(*nodes, x0)
    n = 18                                            # past the slice-15 re-wrap
    x = np.arange(conf.Nx + 3) % conf.Nx * 2 * np.pi / conf.Nx
    hist = np.concatenate([0.3 * np.cos(x + 0.1 * m) for m in range(n + 1)])
    padded = np.concatenate([hist, np.zeros(conf.stride_t() + 8)])
    with nufi.GpuScheduler(conf, conf_metrics=cm) as s:
        s.upload_history(hist, 0, n + 1)
        for m in (0, 1, n):
            got, parts = np.zeros(4), np.zeros(4)
            total = cm.Nx * cm.Nu
            s.compute_metrics(m, 0, total)
            s.download_metrics(got)
            for a, b in ((0, 11), (11, total // 2 + 3), (total // 2 + 3, total)):
                s.compute_metrics(m, a, b)
                s.download_metrics(parts)
            ref = O.metrics(conf, m, padded, conf_metrics=cm)
            err = np.max(np.abs(got - ref) / np.abs(ref))
            print(f"[metrics 1d] {field} {nodes} n={m} max rel err {err:.3e}", flush=True)
            assert err <= 1e-12
            assert np.max(np.abs(parts - got) / np.abs(got)) <= 1e-13
