"""The advections on grids whose state is just below and above the last-level
cache, from where the old and new tendencies are read and written past it:
against the oracle at 1e-12, the bar of operators without a solve.  (The
microphysics' rates of such grids: tests/test_gpu_step_micro.py.)"""
import pytest

import vvm_amd as V
from helpers import assert_fields_close, gpu_run_op, perturbed_state

pytestmark = pytest.mark.gpu

OPS = {"pzeta_pt": (["pzeta_pt"], ["zetap", "dzeta_advect", "dth_buoyancy"]),
       "pscalars": (["pth_pt", "pqv_pt", "pqc_pt", "pqr_pt"],
                    ["thp", "qvp", "qcp", "qrp", "dth_advect", "dqv_advect", "dqc_advect", "dqr_advect", "dqr_VT",
                     "precip"])}


@pytest.mark.parametrize("step", [3, 4])
@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("nx,nz", [(4096, 180), (4096, 200), (4090, 201)])
def test_advection_around_the_cache(oracle, nx, nz, op, step):
    c = V.grid_case(nx, nz)
    st = perturbed_state(c, seed=nx + nz, step=step)
    want = st.copy()
    names, fields = OPS[op]
    for name in names:
        oracle.op(name, c.cfg, want)
    print(f"{op} {nx}x{nz}", flush=True)
    with V.Device(c.cfg) as dev:
        got = gpu_run_op(dev, st, op)
    assert_fields_close(got, want, fields, 1e-12, where=f"{op} {nx}x{nz}")
