"""The one-workgroup field solve over lengths of every kind of stage (factors 2,
3, 4, 5, larger primes, a prime length, short rings) and over the splits of the
partial sums, in 1D and 3D: energy and coefficients of a rho trace against the
oracle, to 1e-12, the bar of the other FP64 parity tests.  The stage list itself
is checked on the CPU."""
import numpy as np
import pytest

import numericalflowiteration_amd as nufi
from numericalflowiteration_amd import config as C
from tests import oracle_lib as O


def radices(L):
    f, rest, p = [], L, 2
    while rest % 4 == 0:
        f.append(4)
        rest //= 4
    while rest > 1:
        if p * p > rest:
            p = rest
        while rest % p == 0:
            f.append(p)
            rest //= p
        p += 1
    return f


def mixed_radix(x):
    """The stages of fft_lds.hpp: mixed_stage, index for index, with its float32 quotients."""
    L, s = x.size, 1
    tw = np.exp(-2j * np.pi * np.arange(L) / L)

    def div(a, y):
        return int((np.float32(a) + np.float32(0.5)) * (np.float32(1) / np.float32(y)))
    for r in radices(L):
        Lr, y = L // r, np.zeros_like(x)
        for o in range(L):
            t = div(o, s)
            assert t == o // s
            q, p = o - t * s, div(t, r)
            assert p == t // r
            k = t - p * r
            m, step, acc = s * k * p, Lr * k, 0j
            assert m < L and step < L
            for j in range(r):
                acc += x[q + s * p + j * Lr] * tw[m]
                m = m + step - (L if m + step >= L else 0)
            y[o] = acc
        x, s = y, s * r
    return x


@pytest.mark.parametrize("L", [3, 6, 10, 12, 15, 20, 49, 97, 100, 120, 242, 360, 1155, 2187, 4374, 5119])
def test_stages_on_the_cpu(L):
    rng = np.random.default_rng(L)
    x = rng.standard_normal(L) + 0j
    if L <= 1200:
        X = np.fft.fft(x)
        assert np.linalg.norm(mixed_radix(x) - X) <= 1e-13 * np.linalg.norm(X)
    f = radices(L)
    assert int(np.prod(f)) == L and len(f) <= 8


def check(name, c, got, h, e, e0):
    """Slices (mean-free, normwise) and energies of steps 0 .. Nt."""
    rows = [np.asarray(a).ravel()[: (c.Nt + 1) * c.stride_t()].reshape(c.Nt + 1, -1) for a in (got, h)]
    g, r = (a - a.mean(axis=1, keepdims=True) for a in rows)
    errs = [np.max(np.linalg.norm(g - r, axis=1) / np.linalg.norm(r, axis=1)), np.max(np.abs(np.asarray(e) - e0) / np.abs(e0))]
    print(f"[field {name}] coefficients {errs[0]:.2e}, energy {errs[1]:.2e}", flush=True)
    assert max(errs) <= 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("Nx,Nu", [(5, 40), (7, 16), (12, 300), (30, 17), (49, 64), (64, 256), (97, 33), (100, 515), (128, 100),
                                   (129, 700), (256, 1030), (360, 40), (600, 33), (1100, 24), (1155, 16)])
def test_field_1d(Nx, Nu):
    c = C.config_1d(Nx, Nu, 1 / 16, 3.5 / 16, 0.0, 4 * np.pi, -8.0, 8.0, C.F0_LANDAU_1D, alpha=0.05, k=0.5)
    h = O.new_history(c, c.Nt + 1)
    e0 = O.run(c, 0, c.Nt + 1, h)
    with nufi.GpuScheduler(c) as s:
        e = s.run()
        got = s.history(0, c.Nt + 1)
    check(f"{Nx}x{Nu}", c, got, h, e, e0)


@pytest.mark.gpu
@pytest.mark.parametrize("N", [(6, 5, 4), (12, 9, 7), (16, 16, 16)])
def test_field_3d(N):
    c = C.config_3d(N, (4, 4, 4), 1 / 8, 2.5 / 8, (0.0, 4 * np.pi), (-6.0, 6.0), C.F0_LANDAU_3D, alpha=0.05, k=0.5)
    h = O.new_history(c, c.Nt + 1)
    e0 = O.run(c, 0, c.Nt + 1, h)
    with nufi.GpuScheduler(c) as s:
        e = s.run()
        got = s.history(0, c.Nt + 1)
    check(N, c, got, h, e, e0)
