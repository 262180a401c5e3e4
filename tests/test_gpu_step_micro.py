"""The timestep's Kessler kernel, which reads the scalars as their advection
left them and applies the negative-value rescale and AddForcing on the way.

Grids whose 64 x 4 tiles (Kessler) and 64 x 8 tiles (advection) are full, have
one column and row more, and are both, one, or none at most 640, up to which
the ratios come from the producer's partial sums instead of k_finalize; and one
row and column past 1024 of the latter, up to which the vorticity's advection
shares their launch (the operators have one each); and 4096 x 200, whose rates
are written past the caches.  One
step with every kind of forcing, negative cloud and a few points of negative
rain (whose fall speed is NaN), against the same phases as separate operators.
The microphysics' rates come straight from that kernel and have to be the same
bits: both routes round alike, operation by operation.  The fields have the
diffusion sweep behind them, in tiles and in order, which differ by 1e-12 at
most."""
import numpy as np
import pytest

import vvm_amd as V
from helpers import perturbed_state

pytestmark = pytest.mark.gpu

PHASES = ["pzeta_pt", "pscalars", "forcing_bc", "pubarTop_pt", "cal_w", "cal_u", "microphysics", "turbulence", "nudge",
          "nextTimeStep"]
RATES = ["evaporation", "accretion", "autoconversion", "condensation", "precip"]


@pytest.mark.parametrize("nx,nz", [(64, 8), (65, 9), (66, 10), (67, 11), (63, 19), (1100, 150), (2100, 170), (2048, 256),
                                   (2049, 257), (4096, 200)])
@pytest.mark.parametrize("forced", [False, True])
def test_step_forcing_and_kessler(nx, nz, forced):
    kw = dict(tropical_forcing=1, addforcingtime=10.0) if forced else {}
    c = V.grid_case(nx, nz, **kw)
    st = perturbed_state(c, seed=nx + nz, step=2)
    rng = np.random.default_rng(nz)
    st["qc"][:] += rng.normal(0, 1e-4, st["qc"].shape)
    st["qr"][:] = np.abs(st["qr"]) - 1e-6
    rate = rng.normal(0.0, 5.0, (c.cfg.nx, c.cfg.nz))
    print(f"step {nx}x{nz} forced {forced}", flush=True)
    got, want = st.copy(), st.copy()
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        if forced:
            dev.set_radiation(rate, True)
        dev.step(1)
        dev.download(got)
    want.step = got.step
    want.status_for_adding_forcing = got.status_for_adding_forcing
    want["init_th_forcing"][:] = got["init_th_forcing"]
    assert want.status_for_adding_forcing == int(forced)
    with V.Device(c.cfg) as dev:
        dev.upload(want)
        if forced:
            dev.set_radiation(rate, True)
        for op in PHASES:
            dev.op(op)
        dev.download(want)
    for f in RATES:
        np.testing.assert_array_equal(got[f], want[f], err_msg=f)
    for f in ("th", "qv", "qc", "qr", "zeta"):
        inner = np.s_[1:-1, 1:-1]
        scale = np.abs(want[f][inner]).max()
        np.testing.assert_allclose(got[f][inner], want[f][inner], rtol=0, atol=1e-12 * scale, err_msg=f)
