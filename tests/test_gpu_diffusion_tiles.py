"""The K-diffusion sweep as independent tiles, and the choice between its
warm-ups (8, 16, 32 columns and rows) and the sweep in order.

The weights a + d of the sweep are at most rho = K dt (1/dx^2 + r/dz^2), r the
largest density ratio; the grid spacing sets which of the four runs.  Grids at
the edges of a tile's columns (55, 47 and 31 stored by one wavefront) and rows
(16 or 32 a wavefront, four wavefronts a workgroup).  Against the oracle's sequential sweep at 1e-12,
the bar of the sweep in order: the tiles differ from it by less than 2^-53 of
the change the sweep makes, and both by the rounding of the sums."""
import numpy as np
import pytest

import vvm_amd as V
from helpers import assert_fields_close, gpu_run_op, perturbed_state

pytestmark = pytest.mark.gpu

FIELDS = ["RKM", "RKH", "zetap", "thp", "qvp", "qcp", "qrp"]


def halo(c, st):
    """The warm-up the coefficients ask for (0: the sweep in order)."""
    k = max(st["RKM"].max(), st["RKH"].max())
    ru, rw = st["rhou"], st["rhow"]
    r = max((ru[:-2] / rw[1:-1]).max(), (rw[1:-1] / ru[1:-1]).max())
    rho = k * c.cfg.dt * (1 / c.cfg.dx ** 2 + r / c.cfg.dz ** 2)
    return next((h for h in (8, 16, 32) if rho <= 2.0 ** (-53 / h)), 0), rho


def state(c, seed, wind):
    st = perturbed_state(c, seed=seed, step=5)
    st["u"][:] *= wind
    st["w"][:] *= wind
    for f in ("zeta", "th", "qv", "qc", "qr"):
        st[f + "p"][:] = st[f]
    return st


# dx, the winds' scale and dt that give each warm-up
REGIMES = {8: (100.0, 0.01, 0.3), 16: (30.0, 0.01, 1.0), 32: (12.0, 0.002, 1.0), 0: (6.0, 0.002, 1.0)}


@pytest.mark.parametrize("want_halo", list(REGIMES))
@pytest.mark.parametrize("nx,nz", [(6, 6), (31, 17), (47, 16), (55, 64), (56, 65), (63, 33), (64, 129), (111, 30),
                                   (300, 70), (1000, 14)])
def test_sweep_matches_oracle(oracle, nx, nz, want_halo):
    dx, wind, dt = REGIMES[want_halo]
    c = V.grid_case(nx, nz, dx=dx, dt=dt)
    st = state(c, nx + nz, wind)
    want = st.copy()
    oracle.op("turbulence", c.cfg, want)
    h, rho = halo(c, want)
    print(f"turbulence {nx}x{nz} dx {dx:g}: rho {rho:.3g}, warm-up {h}", flush=True)
    assert h == want_halo
    with V.Device(c.cfg) as dev:
        got = gpu_run_op(dev, st, "turbulence")
    assert_fields_close(got, want, FIELDS, 1e-12, where=f"turbulence {nx}x{nz} warm-up {h}")
    for f in FIELDS[2:]:  # the ghost cells are not updated
        for edge in (np.s_[0, :], np.s_[-1, :], np.s_[:, 0], np.s_[:, -1]):
            np.testing.assert_array_equal(got[f][edge], want[f][edge], err_msg=f)


@pytest.mark.parametrize("nx,nz,dx", [(96, 40, 100.0), (96, 40, 8.0)])
def test_steps_through_changing_coefficients(oracle, nx, nz, dx):
    """Steps from strong winds, whose coefficients fall from step to step: the
    warm-up guessed from the step before is checked against this step's."""
    c = V.grid_case(nx, nz, dx=dx, dt=0.02 * dx)
    st = perturbed_state(c, seed=3, step=0)
    for f in ("u", "w"):
        st[f][:] *= 0.1
    want = st.copy()
    oracle.step(c.cfg, want, 3)
    print(f"3 steps of {nx}x{nz} at {dx:g} m", flush=True)
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        dev.step(3)
        got = st.copy()
        dev.download(got)
    assert_fields_close(got, want, ["zeta", "zetam", "th", "thm", "qv", "qc", "qr", "u", "w", "RKM", "RKH"], 1e-9,
                        where=f"{nx}x{nz} 3 steps")
