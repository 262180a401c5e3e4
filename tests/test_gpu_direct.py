"""The direct solve of the cal_w system on the GPU (k_direct.hip).

The isolated solve against the oracle's direct method, over column counts
that take every stage of the row transform (radices 8, 4, 2, 3, 5, and the
direct sum for other primes, with its twiddles in LDS or not) and row counts
at the edges of the elimination (even and odd, the smallest and the largest
grid).  A backward-stable solve has a relative error of a few eps times the
condition number of L, here about (M + 1)^2 (largest eigenvalue ~ 8, smallest
~ (pi / (M + 1))^2 in units of the conductances): 32 eps (M + 1)^2 in FP64.
With FP32 corrections the stop rule fixes the residual, so the error is at
most that times the condition number.

The step's solve corrects further where one solve misses the stop rule; a
rule below round-off takes that path.
"""
import numpy as np
import pytest

import vvm_amd as V
from helpers import rel_err

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps
SIZES = [(6, 6), (7, 7), (8, 8), (16, 12), (30, 31), (49, 20), (127, 40), (128, 64), (250, 33), (317, 61),
         (1000, 100), (2048, 256), (3000, 24), (2 * 1021, 9), (4099, 7), (8191, 6), (8192, 6), (24, 478)]
_exact = {}  # the oracle's solutions, one for both modes


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,nz", SIZES)
def test_direct_solve_matches_oracle(oracle, nx, nz, mode):
    over = dict(solver_mode=V.VVM_SOLVER_MIXED, stop_mode=V.VVM_STOP_REL, tol_rel=1e-12) if mode == "mixed" else {}
    c = V.grid_case(nx, nz, dx=50.0, **over)
    st = V.init_state(c)
    n, m = nx, nz - 1
    rng = np.random.default_rng(nx + nz)
    b = rng.normal(0, 1, n * m)
    x = rng.normal(0, 1, n * m)  # a guess that is no help
    if (nx, nz) not in _exact:
        _exact[nx, nz] = oracle.poisson_exact(c.cfg, st["rhou"], st["rhow"], b)
    want = _exact[nx, nz]
    print(f"direct solve {mode} {nx}x{nz}", flush=True)
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        s = dev.poisson(b, x)
        assert dev.last_rc == 0
        again = rng.normal(0, 1, n * m)
        dev.poisson(b, again)
    cond = (m + 1.0) ** 2
    tol = 32 * EPS * cond if mode == "fp64" else 1e-12 * cond
    assert s.rel_residual <= (1e-13 if mode == "fp64" else 1e-12) and 1 <= s.iters <= 8
    assert rel_err(x, want) <= tol, (rel_err(x, want), tol)
    assert rel_err(again, x) <= 2 * tol


@pytest.mark.parametrize("nx,nz", [(128, 64), (49, 21)])
@pytest.mark.parametrize("mode", ["fp64", "mixed"])
def test_step_beyond_round_off(nx, nz, mode):
    """A stop rule below round-off: FP64 accepts the residual it can reach,
    the mixed solver warns, and both give the step that one solve gives."""
    solver = V.VVM_SOLVER_MIXED if mode == "mixed" else V.VVM_SOLVER_FP64
    out = []
    for tol in (1e-10, 1e-18):
        c = V.grid_case(nx, nz, solver_mode=solver, stop_mode=V.VVM_STOP_REL, tol_rel=tol)
        st = V.init_state(c)
        print(f"step {mode} {nx}x{nz} tol {tol:g}", flush=True)
        with V.Device(c.cfg) as dev:
            dev.upload(st)
            s = dev.step(3)
            dev.download(st)
        out.append((st, s))
    (a, sa), (b, sb) = out
    assert sa.not_converged == 0 and sa.solve_iters_total == 3
    assert sb.not_converged == (0 if mode == "fp64" else 3) and sb.solve_iters_total > 3
    for f in ("zeta", "th", "qv", "u", "w"):
        assert rel_err(b[f], a[f]) <= 32 * EPS * nz ** 2, f
