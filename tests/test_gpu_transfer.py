"""The state between host and device (k_transfer.hip), bit for bit.

Grids at the edges of what a workgroup (16 columns, 8 of an AB2 history) and a
slot of pinned memory (1 MiB) take: a state in one piece, fields that straddle
slots, one field over several, the longest and the shortest columns."""
import threading

import numpy as np
import pytest

import vvm_amd as V

pytestmark = pytest.mark.gpu


def random_state(c, seed):
    st = V.init_state(c)
    rng = np.random.default_rng(seed)
    for n in V.FIELDS2D + V.HISTS + V.ROWS:
        st[n][:] = rng.normal(0, 1, st[n].shape)
    return st


@pytest.mark.parametrize("nx,nz", [(6, 6), (14, 9), (15, 10), (62, 476), (130, 64), (317, 61), (700, 130), (2050, 70),
                                   (8190, 14)])
def test_round_trip(nx, nz):
    c = V.grid_case(nx, nz)
    st = random_state(c, nx + nz)
    print(f"state {nx}x{nz} there and back", flush=True)
    with V.Device(c.cfg) as dev:
        for turn in range(2):
            dev.upload(st)
            got = V.HostState(c.cfg.nx, c.cfg.nz)
            dev.download(got)
            for n in st.a:
                np.testing.assert_array_equal(got[n], st[n], err_msg=n)
            st = random_state(c, turn)
        # some arrays only: the others are left alone
        part = V.HostState(c.cfg.nx, c.cfg.nz)
        v = part.view()
        for n in part.a:
            if n not in ("w", "dqr_VT", "precip", "thb"):
                setattr(v, n, None)
        assert dev.lib.vvm_dev_download(dev.h, V.C.byref(v)) == 0
        for n in part.a:
            want = got[n] if n in ("w", "dqr_VT", "precip", "thb") else np.zeros_like(part[n])
            np.testing.assert_array_equal(part[n], want, err_msg=n)


def test_two_handles_at_once():
    """Two threads move the states of their own handles."""
    cases = [V.grid_case(700, 130), V.grid_case(512, 200)]
    states = [random_state(c, 9 + k) for k, c in enumerate(cases)]
    got = [V.HostState(c.cfg.nx, c.cfg.nz) for c in cases]

    def work(k):
        with V.Device(cases[k].cfg) as dev:
            for _ in range(3):
                dev.upload(states[k])
                dev.download(got[k])

    print("two states at once", flush=True)
    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        for n in states[k].a:
            np.testing.assert_array_equal(got[k][n], states[k][n], err_msg=n)
