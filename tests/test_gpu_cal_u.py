"""cal_u: the top row from its prefix sums and the integral below it.

Columns at the edges of a workgroup's 16 and of the 1024 threads' runs (one
value a thread up to 1024 columns, eight at 8192); levels at the edges of the
64 chunks (one level each up to 67 rows) and of the four levels of a chunk that
a thread keeps in registers (up to 259 rows).  At 1e-11, the operator's bar,
against the closed form in extended precision: the oracle's own top row is
1.0e-11 from it at 2047 columns and 2.5e-11 at 8192."""
import numpy as np
import pytest

import vvm_amd as V
from helpers import gpu_run_op, perturbed_state

pytestmark = pytest.mark.gpu


def cal_u(c, st):
    """src/PoissonSolver.cpp:580-653 on the interior, in extended precision."""
    x = {f: st[f].astype(np.longdouble) for f in ("w", "zetap", "rhow", "rhou")}
    n, nz, dx, dz = c.cfg.nx - 2, c.cfg.nz, np.longdouble(c.cfg.dx), np.longdouble(c.cfg.dz)
    h = x["rhow"][nz - 2] * x["w"][1:n + 1, nz - 2] / x["rhou"][nz - 2] * dx
    prefix = np.concatenate([[0], np.cumsum(h - h.mean())[:-1]])
    d = prefix - prefix.mean()
    y = np.cumsum(d)
    u = np.zeros((n, nz), np.longdouble)
    u[:, nz - 2] = d / dx + st.s["ubarTopp"]
    for k in range(nz - 3, 0, -1):
        grad = (x["w"][1:n + 1, k + 1] - x["w"][:n, k + 1]) / dx
        u[:, k] = u[:, k + 1] - dz * (grad - x["rhow"][k + 1] * x["zetap"][1:n + 1, k + 1])
    return u[:, 1:nz - 1], d / dx, y - y.mean()


@pytest.mark.parametrize("nx,nz", [(8, 8), (15, 9), (16, 64), (17, 65), (33, 66), (1024, 12), (1025, 12), (2047, 10),
                                   (8192, 10), (40, 256), (40, 257), (40, 258), (24, 478)])
def test_cal_u(nx, nz):
    c = V.grid_case(nx, nz, dx=20.0)
    st = perturbed_state(c, seed=nx + nz, step=3)
    st["zetap"][:] = st["zeta"]
    print(f"cal_u {nx}x{nz}", flush=True)
    want = cal_u(c, st)
    with V.Device(c.cfg) as dev:
        got = gpu_run_op(dev, st, "cal_u")
    have = got["u"][1:-1, 1:-1], got["uxi"][1:-1], got["xi"][1:-1]
    for name, a, b in zip(("u", "uxi", "xi"), have, want):
        err = float(np.linalg.norm(a - b) / np.linalg.norm(b))
        assert err <= 1e-11, f"{name} of {nx}x{nz}: {err:.2e}"
