"""What vvm_dev_tune chooses from: a launch shape is a candidate only where it
changes a launch, and a result is passed on only between handles that choose
from the same candidates.

The strip width matters where the sweep runs in order (weights 10 dt (1/dx^2 +
1/dz^2) above 0.32, the widest warm-up's bound; 0.56 at 6 m and 1 s), the
coarse budget where MG-PCG solves (FP64 with a guess)."""
import pytest

import vvm_amd as V

pytestmark = pytest.mark.gpu

SHAPE = dict(solver_mode=V.VVM_SOLVER_FP64)
PCG = dict(solver_mode=V.VVM_SOLVER_FP64, guess_mode=V.VVM_GUESS_EXTRAP2, stop_mode=V.VVM_STOP_REL, tol_rel=1e-10)


def tune(nx, nz, dx, over):
    c = V.grid_case(nx, nz, dx=dx, dt=0.01 * dx if dx > 10 else 1.0, **over)
    print(f"tune {nx}x{nz} dx {dx:g} {over}", flush=True)
    with V.Device(c.cfg) as dev:
        dev.upload(V.init_state(c))
        return dev.tune(2)


@pytest.mark.parametrize("nx,nz", [(512, 32), (640, 40), (700, 33)])
def test_default_where_nothing_can_be_chosen(nx, nz):
    r = tune(nx, nz, 100.0, SHAPE)
    assert (r.diffusion_strip_waves, r.mg_coarse_lds_kib) == (4, 64)
    assert r.ms_per_step == r.ms_default > 0.0


def test_results_stay_with_their_candidates():
    direct, pcg, order = (tune(576, 48, dx, over) for dx, over in ((100.0, SHAPE), (100.0, PCG), (6.0, SHAPE)))
    assert (direct.diffusion_strip_waves, direct.mg_coarse_lds_kib) == (4, 64)
    assert pcg.diffusion_strip_waves == 4 and pcg.mg_coarse_lds_kib in (16, 32, 64)
    assert order.diffusion_strip_waves in (2, 4, 8) and order.mg_coarse_lds_kib == 64
    # measured each for itself, not taken over
    assert len({direct.ms_default, pcg.ms_default, order.ms_default}) == 3
    again = tune(576, 48, 100.0, PCG)
    assert (again.mg_coarse_lds_kib, again.ms_default) == (pcg.mg_coarse_lds_kib, pcg.ms_default)
