"""The row transform as a convolution with a chirp, for column counts with large
prime factors.

Primes and multiples of primes at the rule's edges (sums of the factors above 5
of 10 and 28, below and above 1024 columns), just under a power of two (the
shortest padding), the largest convolution (4093 columns) and the first count
past it (4111, summed directly).  As tests/test_gpu_direct.py: 32 eps (M + 1)^2
in FP64, the stop rule times the condition number with FP32 corrections."""
import numpy as np
import pytest

import vvm_amd as V
from helpers import COMPARE_STEP, assert_fields_close, perturbed_state, rel_err

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("nx,nz", [(11, 9), (14, 8), (22, 31), (31, 20), (61, 33), (121, 10), (257, 40), (509, 17),
                                   (511, 64), (1021, 30), (1064, 12), (1111, 9), (1184, 9), (2047, 8), (2053, 12),
                                   (4093, 9), (4111, 7)])
def test_solve_matches_oracle(oracle, nx, nz, mode):
    over = dict(solver_mode=V.VVM_SOLVER_MIXED, stop_mode=V.VVM_STOP_REL, tol_rel=1e-12) if mode == "mixed" else {}
    c = V.grid_case(nx, nz, dx=50.0, **over)
    st = V.init_state(c)
    n, m = nx, nz - 1
    rng = np.random.default_rng(nx + nz)
    b, x = rng.normal(0, 1, n * m), rng.normal(0, 1, n * m)
    want = oracle.poisson_exact(c.cfg, st["rhou"], st["rhow"], b)
    print(f"chirp solve {mode} {nx}x{nz}", flush=True)
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        dev.poisson(b, x)
        assert dev.last_rc == 0
    cond = (m + 1.0) ** 2
    tol = 32 * EPS * cond if mode == "fp64" else 1e-12 * cond
    assert rel_err(x, want) <= tol, (rel_err(x, want), tol)


@pytest.mark.parametrize("nx,nz", [(29, 20), (317, 12), (1021, 70)])
def test_step_matches_oracle(oracle, nx, nz):
    """A step, whose microphysics shares these launches, at the step's 1e-10."""
    c = V.grid_case(nx, nz, stop_mode=V.VVM_STOP_REL, tol_rel=1e-12)
    st = perturbed_state(c, seed=nx, step=2)
    want, got = st.copy(), st.copy()
    print(f"chirp step {nx}x{nz}", flush=True)
    oracle.step(c.cfg, want, 1)
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        dev.step(1)
        dev.download(got)
    assert_fields_close(got, want, COMPARE_STEP, 1e-10, where=f"step {nx}x{nz}")
