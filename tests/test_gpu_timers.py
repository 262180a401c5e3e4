"""What the kernel timer and the step's phase times count: every launch of the
selected kernel, also where the sweep runs in order or a step's end runs twice.
The inputs that lead there are those of test_gpu_redo and
test_gpu_diffusion_order."""
import numpy as np
import pytest

import vvm_amd as V
from helpers import perturbed_state

pytestmark = pytest.mark.gpu

KT_TURB, KT_DIFFUSION, KT_CALU = 5, 6, 8


def test_sweep_in_order_is_timed():
    # K is at least 10: weights of 10 dt (1/dx^2 + 1/dz^2) = 0.56, above the widest warm-up's 0.32
    c = V.grid_case(200, 40, dx=6.0, dt=1.0)
    st = perturbed_state(c, seed=1, step=5)
    for f in ("u", "w", "zeta"):
        st[f][:] *= 0.002
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        dev.kernel_timer(KT_DIFFUSION)
        dev.step(1)
        first = dev.kernel_time()[1]  # the first step may have queued tiles before it knew
        dev.step(3)
        avg, n = dev.kernel_time()
    assert first >= 1 and n == first + 3 and avg > 0.0


@pytest.mark.parametrize("kernel", [KT_TURB, KT_DIFFUSION, KT_CALU])
def test_repeated_launches_are_timed(kernel):
    """A rule below round-off: the first step's solve is corrected after what
    follows it has been queued, which then runs again."""
    c = V.grid_case(128, 64, stop_mode=V.VVM_STOP_REL, tol_rel=1e-18)
    with V.Device(c.cfg) as dev:
        dev.upload(V.init_state(c))
        dev.kernel_timer(kernel)
        s = dev.step(1)
        _, n = dev.kernel_time()
    assert s.solve_iters_last > 1 and n == 2


def test_ensemble_members_are_timed():
    """A member's timers count the ensemble's steps as calls of one step."""
    cases = [V.grid_case(64, 32, seed=k) for k in range(3)]
    steps = 300  # more than the kernel timer holds between two readings
    times = np.zeros((2, 5))
    with V.Ensemble(cases, threads=2) as ens:
        a, b = ens.member(0), ens.member(1)
        a.kernel_timer(KT_CALU)
        b._check(b.lib.vvm_dev_set_step_timers(b.h, times.ctypes.data_as(V.PTR), 2), "set_step_timers")
        ens.step(0)
        assert not times.any()
        ens.step(steps)
        avg, n = a.kernel_time()
        assert n == steps and avg > 0.0
        assert (times[0] > 0.0).all() and not times[1].any()
        assert times[0, :4].max() <= times[0, 4]


def test_phases_of_a_repeated_end():
    """What a correction repeats belongs to the phase of turbulence and
    diffusion, with the kernels' clocks as with events."""
    c = V.grid_case(128, 64, stop_mode=V.VVM_STOP_REL, tol_rel=1e-18)
    st = V.init_state(c)
    for timed in (False, True):
        with V.Device(c.cfg) as dev:
            dev.upload(st)
            s = dev.step_timed(1)[0] if timed else dev.step(1)
        print(f"events {timed}: poisson {s.t_poisson * 1e6:.0f} us, diffusion {s.t_diffusion * 1e6:.0f} us", flush=True)
        assert s.solve_iters_last > 1
        assert 0.0 < s.t_poisson < s.t_diffusion
        assert s.t_advection > 0.0 and s.t_microphysics > 0.0
