"""Sweeps whose waves exchange two neighbours of every unknown through LDS (BCC's rings of four, the
unknown fastest) against the same sweeps without it (the segment fastest, flag 1) and the oracle:
every lane form, lines of one and several waves, a remainder of rows in the last tile, boxes whose
last workgroups are partly empty, and the reverse sweep.

Tolerance: the two traversals add an unknown's neighbours in the same order in the same precision;
they may differ by the compiler's choice of fused operations, a few eps an update, which 8 steps of
a stable scheme grow by less than 50."""
import numpy as np
import pytest

from helpers import oracle_params, random_state, rel_l2, with_field
from oracle_lib import Oracle
from spacetime_amd import gpe, lattice

pytestmark = pytest.mark.gpu

FIELD = dict(bq=4e-3, bb=(0.01, -0.02, 0.05))
BOXES = [(3, gpe.FP32, (130, 9, 3), 2), (5, gpe.FP32, (130, 5, 2), 1), (3, gpe.FP32, (300, 3, 2), 2),
         (5, gpe.FP32, (34, 13, 3), 2), (3, gpe.FP64, (96, 11, 3), 1), (5, gpe.FP64, (65, 4, 2), 1),
         (3, gpe.FP64, (128, 3, 5), 1), (3, gpe.FP32, (1, 1, 1), 2)]


@pytest.mark.parametrize("ncomp,precision,dims,xpl", BOXES)
def test_exchange_equals_plain_sweeps(ncomp, precision, dims, xpl):
    cfg = gpe.Config.centred_box("bcc", dims, 0.7, ncomp=ncomp, precision=precision, dt=2e-4, c0=60.0, c1=8.0, c2=3.0,
                                 q=0.1)
    eps = 2.0 ** -52 if precision == gpe.FP64 else 2.0 ** -23
    psi0, target = random_state(cfg.shape, 3), random_state(cfg.shape, 4)
    got = []
    for flags in (1, 3):
        with gpe.Stepper(cfg) as st:
            st.set_traversal(8, flags, xpl)
            st.set_field(**FIELD)
            st.set_state(psi0)
            st.start(gpe.START_EULER)
            st.step(8)
            out = [st.get_state(0)]
            st.set_state(psi0)
            st.itp(3, 1e-4)
            out.append(st.get_state(0))
            st.set_state(psi0)
            res = st.adjoint(7, 3, gpe.OBJ_OVERLAP, target)
            out.append(np.array([res["J"]] + list(res["grad_trap"]) + list(res["grad_static_bb"])))
            got.append(out)
    for plain, ring in zip(*got):
        assert rel_l2(ring, plain) < 50 * 8 * eps
    o = Oracle()
    L, p = o.lattice(lattice.get("bcc")), with_field(oracle_params(o, cfg), **FIELD)
    a = psi0.copy()
    b = o.forward_euler(L, p, a, cfg.dt)
    o.leapfrog3(L, p, a, b, cfg.dt, 8, t0=cfg.dt)
    assert rel_l2(got[1][0], b) < 50 * 8 * eps
