"""The adjoint over every shape of its segments (one sweep, one segment, a last segment of one or two
levels, intervals longer than the run) on one context whose workspace is reused, grown and found
stale: recomputed levels carry the same bits as stored ones, so every interval gives the same
objective, gradients and final levels."""
import numpy as np
import pytest

from helpers import random_state
from spacetime_amd import gpe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,fp64", [(gpe.FP32, False), (gpe.FP64, False), (gpe.FP32, True)])
@pytest.mark.parametrize("objective", [gpe.OBJ_OVERLAP, gpe.OBJ_ENERGY, gpe.OBJ_MAGNETIZATION_Z])
def test_intervals_agree(precision, fp64, objective):
    cfg = gpe.Config.centred_box("bcc", (9, 6, 5), 0.6, ncomp=3, precision=precision, dt=2e-4, c0=60.0, c1=8.0, q=0.1)
    psi0, target = random_state(cfg.shape, 1), random_state(cfg.shape, 2)

    def run(st, nsweeps, every):
        st.set_knot_ramp([0.02, -0.05, 0.03], 10 * cfg.dt, 4e-3)
        st._ramp_sizes = (1, 3)
        st.set_state(psi0)
        r = st.adjoint(nsweeps, every, objective, target if objective == gpe.OBJ_OVERLAP else None, fp64)
        return [np.array([r["J"]]), r["grad_trap"], r["grad_ramp_b"], st.get_state(0), st.get_state(1)]

    with gpe.Stepper(cfg) as kept:
        for nsweeps, intervals in ((1, (2, 5)), (2, (2, 3)), (9, (2, 3, 4, 8, 9, 20)), (13, (12, 6, 13))):
            with gpe.Stepper(cfg) as fresh:
                expect = run(fresh, nsweeps, nsweeps + 3)
            for every in intervals:
                for got, ref in zip(run(kept, nsweeps, every), expect):
                    np.testing.assert_array_equal(got, ref, err_msg="%d sweeps, every %d" % (nsweeps, every))
