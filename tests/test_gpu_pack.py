"""States into the device layout and back: runs of cells from 16 to 1024 a workgroup, a partial last
run, runs over several rows and planes, every cell size, lines padded and not.  The way back through
the chunked fetch is a kernel of its own.  A copy is exact: FP64 bits, FP32 once rounded."""
import ctypes

import numpy as np
import pytest

from helpers import random_state
from spacetime_amd import gpe

pytestmark = pytest.mark.gpu

BOXES = [("cube", 1, (1, 1, 1)), ("cube", 1, (1, 37, 5)), ("cube", 1, (128, 100, 90)), ("cube", 5, (75, 31, 9)),
         ("bcc", 3, (8, 6, 5)), ("bcc", 1, (129, 33, 40)), ("fcc", 3, (41, 40, 21)), ("a15", 5, (17, 3, 11)),
         ("c15", 3, (57, 9, 2)), ("c15", 1, (30, 29, 23)), ("fcc", 3, (61, 61, 61)), ("z", 5, (34, 5, 3))]


@pytest.mark.parametrize("precision", [gpe.FP32, gpe.FP64])
@pytest.mark.parametrize("lat,ncomp,dims", BOXES)
def test_there_and_back(lat, ncomp, dims, precision):
    cfg = gpe.Config.centred_box(lat, dims, 0.7, ncomp=ncomp, precision=precision, dt=1e-4)
    psi = random_state(cfg.shape, 9)
    want = psi if precision == gpe.FP64 else psi.astype(np.complex64).astype(np.complex128)
    with gpe.Stepper(cfg) as st:
        st.set_state(psi)
        np.testing.assert_array_equal(st.get_state(0), want)
        back = np.zeros(cfg.shape, np.complex128)
        f = st.lib.gpe_get_state_noalloc
        f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p]
        f.restype = ctypes.c_int
        assert f(st._h, 0, back.ctypes.data) == 0
        np.testing.assert_array_equal(back, want)
