"""Layout changes on both sides of the lines between the two kernels, and the one through LDS over planes
shorter than a workgroup's run of cells.  A copy is exact: FP64 bits, FP32 once rounded."""
import numpy as np
import pytest

from helpers import random_state
from spacetime_amd import gpe

pytestmark = pytest.mark.gpu

BOXES = [("bcc", 1, (28, 26, 30)), ("bcc", 1, (28, 26, 31)),     # 262080 and 270816 values (the line in: 262144)
         ("z", 3, (13, 12, 14)), ("c15", 1, (16, 15, 16)),       # 524160 and 522240 (the line out: 524288)
         ("z", 3, (13, 14, 13)), ("c15", 1, (16, 15, 17)),       # 567840 and 554880
         ("a15", 5, (3, 2, 400)), ("z", 3, (1, 1, 2300)), ("c15", 1, (7, 3, 190)), ("fcc", 5, (5, 7, 300)),
         ("bcc", 3, (61, 62, 61)), ("bcc", 3, (63, 62, 61)),     # 8305272 and 8577576 (2^23 = 8388608)
         ("a15", 1, (57, 57, 57)), ("a15", 3, (43, 39, 37))]     # 8518878 and 8562762


@pytest.mark.parametrize("precision", [gpe.FP32, gpe.FP64])
@pytest.mark.parametrize("lat,ncomp,dims", BOXES)
def test_there_and_back(lat, ncomp, dims, precision):
    cfg = gpe.Config.centred_box(lat, dims, 0.7, ncomp=ncomp, precision=precision, dt=1e-4)
    psi = random_state(cfg.shape, 9)
    want = psi if precision == gpe.FP64 else psi.astype(np.complex64).astype(np.complex128)
    with gpe.Stepper(cfg) as st:
        st.set_state(psi)
        np.testing.assert_array_equal(st.get_state(0), want)
