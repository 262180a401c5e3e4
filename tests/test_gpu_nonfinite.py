"""A value that is not finite in a diffused field reaches every point to its
east and above in one sweep, as in the sequential loop, whether the other
points' weights would let the sweep run as tiles or not: the same points are
finite as in the oracle, and equal to its values at 1e-12."""
import numpy as np
import pytest

import vvm_amd as V
from helpers import gpu_run_op, perturbed_state

pytestmark = pytest.mark.gpu

FIELDS = {"zeta": "zetap", "th": "thp", "qv": "qvp", "qc": "qcp", "qr": "qrp"}


def tile_state(nx, nz):
    """Weights for the tiles with a warm-up of 8."""
    c = V.grid_case(nx, nz, dx=100.0, dt=0.3)
    st = perturbed_state(c, seed=nx + nz, step=5)
    st["u"][:] *= 0.01
    st["w"][:] *= 0.01
    for f, p in FIELDS.items():
        st[p][:] = st[f]
    return c, st


def same(got, want, names, tol):
    for f in names:
        a, b = got[f], want[f]
        fin = np.isfinite(b)
        np.testing.assert_array_equal(np.isfinite(a), fin, err_msg=f)
        assert np.linalg.norm(a[fin] - b[fin]) <= tol * max(np.linalg.norm(b[fin]), 1e-300), f


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("where", [(60, 20), (1, 1), (0, 10), (30, 0)])
@pytest.mark.parametrize("field", list(FIELDS))
def test_operator_carries_it(oracle, field, where, bad):
    c, st = tile_state(200, 60)
    st[FIELDS[field]][where] = bad
    want = st.copy()
    oracle.op("turbulence", c.cfg, want)
    assert not np.isfinite(want[FIELDS[field]][70:-1, 40:-1]).any()  # far beyond the tiles' warm-up
    print(f"turbulence with {bad} in {field} at {where}", flush=True)
    with V.Device(c.cfg) as dev:
        got = gpu_run_op(dev, st, "turbulence")
    same(got, want, FIELDS.values(), 1e-12)


@pytest.mark.parametrize("field", ["th", "zeta"])
def test_step_carries_it(oracle, field):
    c, st = tile_state(200, 60)
    st[field][60, 20] = np.nan
    want = st.copy()
    oracle.step(c.cfg, want, 1)
    print(f"step with NaN in {field}", flush=True)
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        dev.step(1)
        got = st.copy()
        dev.download(got)
    assert not np.isfinite(want[field][80:-1, 40:-1]).any()
    # the negative-value pass makes qv, qc and qr finite first (and not by the same rule as the oracle's)
    for f in ("zeta", "th"):
        np.testing.assert_array_equal(np.isfinite(got[f]), np.isfinite(want[f]), err_msg=f)
