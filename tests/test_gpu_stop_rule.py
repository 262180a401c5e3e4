"""The FP64 solver's stop rules at round-off: VVM_STOP_PARITY goes on until the
residual no longer decreases, whatever one direct solve leaves, and a residual
that cannot decrease counts as converged on every right-hand side.

The right-hand sides are smooth, where round-off is far above 2^-53 of ||b||:
k^-3 vorticity and the lowest mode.  Reference: the same system solved here in
80-bit arithmetic (direct solves in 64 bits, residuals in 80, until they stay).
A solution at the residual's floor is the exact one to a few roundings: 8 eps.
"""
import numpy as np
import pytest

import vvm_amd as V
from helpers import rel_err

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
LD = np.longdouble


def k3_rhs(nx, nz, st, dx, seed):
    """cal_w's right-hand side of a k^-3 vorticity field, rows k = 2 .. nz."""
    rng = np.random.default_rng(seed)
    kx, kz = np.fft.rfftfreq(nx)[None, :], np.fft.fftfreq(nz)[:, None]
    kk = np.sqrt(kx * kx + kz * kz)
    kk[0, 0] = np.inf
    z = np.fft.irfft2(np.fft.rfft2(rng.standard_normal((nz, nx))) * kk ** -1.5, s=(nz, nx))[1:]
    return np.ascontiguousarray(st["rhow"][2:nz + 1, None] ** 2 * (np.roll(z, -1, axis=1) - z) * dx).ravel()


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


@pytest.mark.parametrize("nx,nz", [(512, 64), (512, 256), (317, 61), (2048, 31)])
def test_parity_solve_reaches_the_floor(nx, nz):
    c = V.grid_case(nx, nz)
    st = V.init_state(c)
    b = k3_rhs(nx, nz, st, c.cfg.dx, nx + nz)
    want = exact(st, b, nx)
    print(f"parity solve {nx}x{nz}", flush=True)
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        x = np.zeros_like(b)
        dev.poisson(b, x)
        assert dev.last_rc == 0
        assert rel_err(x, want) <= 8 * EPS
        # a guess good to 1e-13 or so is polished, not returned
        guess = want * (1 + 1e-13 * np.random.default_rng(1).standard_normal(want.size))
        dev.poisson(b, guess)
        assert dev.last_rc == 0
        assert rel_err(guess, want) <= 8 * EPS


@pytest.mark.parametrize("nx,nz", [(512, 64), (317, 61)])
def test_parity_step_operator_reaches_the_floor(nx, nz):
    """cal_w on the same kind of field, w = x / rhow."""
    c = V.grid_case(nx, nz)
    st = V.init_state(c)
    b = k3_rhs(nx, nz, st, c.cfg.dx, nx - nz)
    k = np.arange(2, nz + 1)
    # zetap whose differences along x are b's: its prefix sums
    d = (b.reshape(-1, nx) / (st["rhow"][k, None] ** 2 * c.cfg.dx)).T
    zp = st["zetap"]
    zp[:] = 0.0
    zp[2:-1, 2:nz + 1] = np.cumsum(d, axis=0)[:-1]
    zp[-1, 2:nz + 1] = zp[1, 2:nz + 1]
    zp[0, 2:nz + 1] = zp[-2, 2:nz + 1]
    b = (st["rhow"][k] ** 2 * (zp[2:, k] - zp[1:-1, k]) * c.cfg.dx).T.ravel()
    want = exact(st, b, nx).reshape(-1, nx) / st["rhow"][k, None]
    print(f"parity cal_w {nx}x{nz}", flush=True)
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        dev.op("cal_w")
        dev.download(st)
    assert rel_err(st["w"][1:-1, 2:nz + 1].T, want) <= 8 * EPS


def test_parity_steps_of_a_smooth_flow():
    """The warm bubble's right-hand side, of which one solve leaves 7e-15."""
    c = V.case("c0")
    st = V.init_state(c)
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        s = dev.step(2)
        assert s.not_converged == 0
        assert s.rel_residual_last <= 1e-15 or s.solve_iters_last > 1


def test_queued_correction_gives_the_same_step():
    """A step behind one that needed a correction queues its own; one on a fresh
    handle is corrected after the fact, and one whose first solve was enough
    takes the correction back: the same bits."""
    smooth, rough = V.case("c0"), V.grid_case(128, 64, dx=200.0, dt=2.0)
    fields = ("u", "w", "xi", "uxi")
    with V.Device(smooth.cfg) as dev:
        for c, before in ((smooth, smooth), (rough, smooth), (smooth, rough)):
            st, first = V.init_state(c), V.init_state(before)
            with V.Device(smooth.cfg) as fresh:
                fresh.upload(st)
                s_want = fresh.step(1)
                want = st.copy()
                fresh.download(want)
            dev.upload(first)
            dev.step(1)
            dev.upload(st)
            s = dev.step(1)
            got = st.copy()
            dev.download(got)
            print(f"{before.name} then {c.name}: {s.solve_iters_last} solves, residual {s.rel_residual_last:.1e}",
                  flush=True)
            assert s.solve_iters_last == s_want.solve_iters_last == (2 if c is smooth else 1)
            assert s.refine_last == s_want.refine_last
            np.testing.assert_allclose(s.rel_residual_last, s_want.rel_residual_last, rtol=1e-6)
            for f in fields + ("zeta", "th", "qv", "RKM"):
                np.testing.assert_array_equal(got[f], want[f], err_msg=f)


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
    assert rel_err(x, want) <= (8 * EPS if not stop else 32 * EPS * nz ** 2)
