"""Handles of different grids alive at once: the second one's plan (fewer
columns, less LDS) leaves the first one's launches as they are.  Against the
same solve on a handle that is alone: the same bits."""
import numpy as np
import pytest

import vvm_amd as V

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first,second", [((4096, 16), (2048, 300)), ((6, 470), (8192, 12)), ((3000, 12), (2100, 477))])
def test_two_plans_alive(first, second):
    cases = [V.grid_case(*g, dx=50.0) for g in (first, second)]
    states = [V.init_state(c) for c in cases]
    rhs = [np.random.default_rng(k).standard_normal(g[0] * (g[1] - 1)) for k, g in enumerate((first, second))]
    alone = []
    for c, st, b in zip(cases, states, rhs):
        print(f"solve {c.name} alone", flush=True)
        with V.Device(c.cfg) as dev:
            dev.upload(st)
            x = np.zeros_like(b)
            dev.poisson(b, x)
            alone.append(x)
    with V.Device(cases[0].cfg) as a, V.Device(cases[1].cfg) as b2:
        a.upload(states[0])
        b2.upload(states[1])
        for dev, b, want in ((a, rhs[0], alone[0]), (b2, rhs[1], alone[1]), (a, rhs[0], alone[0])):
            x = np.zeros_like(b)
            dev.poisson(b, x)
            np.testing.assert_array_equal(x, want)
