"""The K-diffusion sweep in order, which coefficients above the tiles' largest
warm-up take, at every strip width that can be set and on wide grids; and the
tiles at their own edges.

The weights a + d of the sweep are at most rho = K dt (1/dx^2 + r/dz^2), r the
largest density ratio; the grid spacing sets which sweep runs, and each test
first asserts that it is the one it is for.

In order: strips of 2, 4 or 8 wavefronts of 64 columns, with whole and partial
last strips, and the one-workgroup sweep of grids narrower than two strips (and
every strip boundary one column off).  Tiles with a warm-up of H columns store
126 - H columns a window (ghost columns included) and H, 8, 16 or 24 rows a
wavefront (32 for H = 32), four wavefronts of them a workgroup for zeta: grids
whose last window holds everything, one column (a ghost) or two, and rows at
these numbers and one off.

Against the oracle's sequential sweep at 1e-12, the bar of both sweeps."""
import numpy as np
import pytest

import vvm_amd as V
from helpers import assert_fields_close, gpu_run_op, perturbed_state

pytestmark = pytest.mark.gpu

FIELDS = ["RKM", "RKH", "zetap", "thp", "qvp", "qcp", "qrp"]
# dx, the winds' scale and dt that give each warm-up (0: in order)
REGIMES = {8: (100.0, 0.01, 0.3), 16: (30.0, 0.01, 1.0), 32: (12.0, 0.002, 1.0), 0: (6.0, 0.002, 1.0)}


def halo(c, st):
    """The warm-up the coefficients ask for (0: the sweep in order)."""
    k = max(st["RKM"].max(), st["RKH"].max())
    ru, rw = st["rhou"], st["rhow"]
    r = max((ru[:-2] / rw[1:-1]).max(), (rw[1:-1] / ru[1:-1]).max())
    rho = k * c.cfg.dt * (1 / c.cfg.dx ** 2 + r / c.cfg.dz ** 2)
    return next((h for h in (8, 16, 32) if rho <= 2.0 ** (-53 / h)), 0)


def check_sweep(oracle, nx, nz, want_halo, cw=0):
    dx, wind, dt = REGIMES[want_halo]
    c = V.grid_case(nx, nz, dx=dx, dt=dt)
    st = perturbed_state(c, seed=nx + nz + cw, step=5)
    st["u"][:] *= wind
    st["w"][:] *= wind
    for f in ("zeta", "th", "qv", "qc", "qr"):
        st[f + "p"][:] = st[f]
    want = st.copy()
    oracle.op("turbulence", c.cfg, want)
    assert halo(c, want) == want_halo
    print(f"turbulence {nx}x{nz} warm-up {want_halo} strips of {cw or 'default'}", flush=True)
    with V.Device(c.cfg) as dev:
        if cw:
            dev.set_strip_waves(cw)
        got = gpu_run_op(dev, st, "turbulence")
    assert_fields_close(got, want, FIELDS, 1e-12, where=f"turbulence {nx}x{nz} warm-up {want_halo} cw {cw}")
    for f in FIELDS[2:]:  # the ghost cells are not updated
        for edge in (np.s_[0, :], np.s_[-1, :], np.s_[:, 0], np.s_[:, -1]):
            np.testing.assert_array_equal(got[f][edge], want[f][edge], err_msg=f)


@pytest.mark.parametrize("cw", [2, 4, 8])
@pytest.mark.parametrize("nx,nz", [(1000, 40), (512, 17), (513, 9), (1023, 12), (2048, 24), (3000, 16)])
def test_strips_in_order(oracle, nx, nz, cw):
    check_sweep(oracle, nx, nz, 0, cw)


@pytest.mark.parametrize("nx", [63, 64, 65, 127, 128, 129, 255, 256, 257])
def test_sweep_in_order_at_strip_edges(oracle, nx):
    check_sweep(oracle, nx, 20, 0)


@pytest.mark.parametrize("want_halo", [8, 16, 32])
@pytest.mark.parametrize("off", [-1, 0, 1, 2])
@pytest.mark.parametrize("windows", [1, 2])
def test_tiles_at_window_edges(oracle, windows, off, want_halo):
    check_sweep(oracle, windows * (126 - want_halo) + off - 2, 20, want_halo)


@pytest.mark.parametrize("want_halo", [8, 16, 32])
@pytest.mark.parametrize("rows", [8, 9, 16, 17, 24, 25, 32, 33, 64, 65, 96, 97, 128, 129])
def test_tiles_at_row_edges(oracle, rows, want_halo):
    check_sweep(oracle, 130, rows, want_halo)


@pytest.mark.parametrize("nx,nz", [(8000, 60), (3000, 200), (1500, 201), (4096, 97)])
def test_tiles_of_more_rows(oracle, nx, nz):
    """More than a workgroup a CU at 8 rows a wavefront: 16 and 24 of them."""
    check_sweep(oracle, nx, nz, 8)


def unstable_row(row, cols):
    """Coefficients that are large in some columns of one row alone: stable
    stratification (K at its smallest, 10) but for a layer turned over there."""
    c = V.grid_case(300, 60, dx=100.0, dt=4.0)
    st = perturbed_state(c, seed=row, step=5)
    for f in ("u", "w", "RKM", "RKH"):
        st[f][:] *= 1e-6
    st["th"][:] = (300.0 + 0.4 * np.arange(st.nz))[None, :]
    st["th"][cols, row - 1] += 60.0
    st["th"][cols, row + 1] -= 60.0
    for f in ("zeta", "th", "qv", "qc", "qr"):
        st[f + "p"][:] = st[f]
    return c, st


# whole rows, single columns, and all columns of the coefficients' 64-wide tiles
# but their first
COLUMNS = {"all": list(range(302)), "inner": [i for i in range(1, 301) if i % 64 != 1], "second": list(range(66, 129)),
           "1": [1], "65": [65], "128": [128], "300": [300]}


@pytest.mark.parametrize("cols", list(COLUMNS))
@pytest.mark.parametrize("row", [1, 2, 16, 17, 18, 33, 49, 60])
def test_warm_up_sees_every_coefficient(oracle, row, cols):
    """The largest coefficient decides, whichever row and columns it is in."""
    cols = COLUMNS[cols]
    c, st = unstable_row(row, cols)
    want = st.copy()
    oracle.op("turbulence", c.cfg, want)
    k = want["RKH"].copy()
    k[cols, row] = 0.0
    k = k[1:-1, 1:-1]  # the ghost cells repeat it
    small = halo(c, {"rhou": want["rhou"], "rhow": want["rhow"], "RKM": k, "RKH": k})
    need = halo(c, want)
    print(f"turned over at row {row}, {len(cols)} columns: warm-up {need}, {small} without it", flush=True)
    assert small == 8 and need != 8
    with V.Device(c.cfg) as dev:
        got = gpu_run_op(dev, st, "turbulence")
    assert_fields_close(got, want, FIELDS, 1e-12, where=f"row {row}, {len(cols)} columns")
