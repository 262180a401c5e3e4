"""The FP64 solver's stop rules at round-off: a residual that cannot decrease
counts as converged on every right-hand side.

The right-hand side is the lowest mode, where round-off is far above 2^-53 of
||b||.  Reference: the same system solved here in 80-bit arithmetic (direct
solves in 64 bits, residuals in 80, until they stay).
"""
import numpy as np
import pytest

import vvm_amd as V
from helpers import rel_err

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
LD = np.longdouble


def exact(st, b, nx):
    """x of L x = -b / rhow, in 80 bits."""
    b = b.reshape(-1, nx)
    m = b.shape[0]
    rhou, rhow = st["rhou"].astype(LD), st["rhow"].astype(LD)
    cx, cu = (1 / rhow[2:2 + m])[:, None], (1 / rhou[1:2 + m])[:, None]
    lam = 4 * np.sin(np.pi * np.arange(nx // 2 + 1) / nx) ** 2
    c = cu.astype(float)
    p = cx.astype(float) * lam + c[1:] + c[:-1]
    for j in range(1, m):
        p[j] -= c[j] * c[j] / p[j - 1]

    def solve(r):
        s = np.fft.rfft(r.astype(float), axis=1)
        for j in range(1, m):
            s[j] += c[j] / p[j - 1] * s[j - 1]
        s[m - 1] /= p[m - 1]
        for j in range(m - 2, -1, -1):
            s[j] = (s[j] + c[j + 1] * s[j + 1]) / p[j]
        return np.fft.irfft(s, n=nx, axis=1)

    f, x = -b.astype(LD) / rhow[2:2 + m, None], np.zeros((m, nx), LD)
    zero = np.zeros((1, nx), LD)
    for _ in range(5):
        up, dn = np.vstack([x[1:], zero]), np.vstack([zero, x[:-1]])
        lx = cx * (2 * x - np.roll(x, 1, 1) - np.roll(x, -1, 1)) + cu[1:] * (x - up) + cu[:-1] * (x - dn)
        x = x + solve(f - lx)
    return x.astype(float).ravel()


@pytest.mark.parametrize("stop", [dict(), dict(stop_mode=V.VVM_STOP_REL, tol_rel=1e-13)])
@pytest.mark.parametrize("nx,nz,dx", [(2048, 256, 100.0), (64, 478, 50.0), (1021, 200, 100.0)])
def test_lowest_mode_converges(nx, nz, dx, stop):
    """Round-off is 1e-12 of ||b|| and more there: the solve ends as converged,
    with the solution the rounding allows (condition number below 32 nz^2)."""
    c = V.grid_case(nx, nz, dx=dx, **stop)
    st = V.init_state(c)
    b = (np.sin(np.pi * np.arange(1, nz) / nz)[:, None] * np.cos(2 * np.pi * np.arange(nx) / nx)[None, :]).ravel()
    want = exact(st, b, nx)
    x = np.zeros_like(b)
    print(f"lowest mode {nx}x{nz} {stop}", flush=True)
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        s = dev.poisson(b, x)
        assert dev.last_rc == 0, s.rel_residual
    assert rel_err(x, want) <= 32 * EPS * nz ** 2
