"""A download into host arrays that share memory: the array that the view lists
last is the one that stays, as if they were copied one after the other."""
import ctypes as C

import numpy as np
import pytest

import vvm_amd as V
from helpers import perturbed_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nz", [(16, 12), (300, 40), (2048, 64)])
def test_last_listed_array_stays(nx, nz):
    c = V.grid_case(nx, nz)
    st = perturbed_state(c, seed=nx, step=3)
    n = st["zeta"].size
    with V.Device(c.cfg) as dev:
        dev.upload(st)
        for names in (("zeta", "zetam", "th"), ("qc", "qr", "u", "w"), ("qv", "dqr_VT")):
            buf = np.zeros(2 * n)
            v = V.VvmHostView()
            for f in names:  # in the view's order; two fields half across the next
                setattr(v, f, buf.ctypes.data_as(V.PTR))
            shifted = names[0] == "qc"
            if shifted:
                v.w = (buf[n // 2:]).ctypes.data_as(V.PTR)
            print(f"{nx}x{nz} {names}", flush=True)
            assert dev.lib.vvm_dev_download(dev.h, C.byref(v)) == 0
            if shifted:
                np.testing.assert_array_equal(buf[:n // 2], st["u"].ravel()[:n // 2])
                np.testing.assert_array_equal(buf[n // 2:n // 2 + n], st["w"].ravel())
            else:
                last = st[names[-1]].ravel()
                np.testing.assert_array_equal(buf[:last.size], last)
