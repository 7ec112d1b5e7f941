"""The adjoint's kept workspace on the device: given back on request, and the next call the same."""
import ctypes

import numpy as np
import pytest

from helpers import random_state
from spacetime_amd import gpe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp64", [False, True])
def test_release_gives_the_memory_back_and_changes_no_bit(fp64):
    cfg = gpe.Config.centred_box("bcc", (40, 40, 40), 0.6, ncomp=3, precision=gpe.FP32, dt=2e-4, c0=60.0, c1=8.0, q=0.1)
    psi0, target = random_state(cfg.shape, 1), random_state(cfg.shape, 2)

    def free():
        avail, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert gpe.load_library().hipMemGetInfo(ctypes.byref(avail), ctypes.byref(total)) == 0  # the runtime it links
        return avail.value

    def run(st):
        st.set_state(psi0)
        r = st.adjoint(12, 8, gpe.OBJ_OVERLAP, target, fp64)
        return [np.array([r["J"]]), r["grad_trap"], r["grad_static_bb"], st.get_state(0), st.get_state(1)]

    with gpe.Stepper(cfg) as st:
        first = run(st)
        kept = free()
        st.release_workspace()
        assert free() - kept > 12 * 8 * 3 * 12 * 40 ** 3  # levels of the run, at least
        for a, b in zip(run(st), first):
            np.testing.assert_array_equal(a, b)
        for a, b in zip(run(st), first):
            np.testing.assert_array_equal(a, b)
