"""FP64 sweeps whose waves pack the rows of a tile (lines that one row a wave would leave partly
idle): boxes with several tiles and a remainder of rows, groups of one and of several waves, lines
just under and over a wave, every sweep mode, the batched launch and the reverse sweep.

Tolerance: the sweeps are the oracle's formula in FP64; 12 steps of a stable scheme grow the
rounding of one (~1e-15 relative) by less than 100."""
import numpy as np
import pytest

from helpers import oracle_params, random_state, rel_l2, with_field
from oracle_lib import Oracle
from spacetime_amd import gpe, lattice

pytestmark = pytest.mark.gpu

FIELD = dict(bq=4e-3, bb=(0.01, -0.02, 0.05))


@pytest.fixture(scope="module")
def oracle():
    return Oracle()


def _run(lat, ncomp, dims):
    return gpe.Config.centred_box(lat, dims, 0.7, ncomp=ncomp, precision=gpe.FP64, dt=2e-4, c0=60.0, c1=8.0, c2=3.0,
                                  q=0.1 if ncomp > 1 else 0.0)


BOXES = [("cube", 1, (65, 9, 3)), ("cube", 3, (7, 41, 3)), ("bcc", 3, (33, 17, 4)), ("bcc", 1, (96, 8, 2)),
         ("fcc", 5, (12, 10, 3)), ("a15", 1, (30, 11, 2)), ("c15", 3, (9, 25, 2)), ("z", 5, (5, 1, 4))]


@pytest.mark.parametrize("lat,ncomp,dims", BOXES)
def test_steps_and_imaginary_time(oracle, lat, ncomp, dims):
    cfg = _run(lat, ncomp, dims)
    L, p = oracle.lattice(lattice.get(lat)), with_field(oracle_params(oracle, cfg), **FIELD)
    psi0 = random_state(cfg.shape, 3)
    with gpe.Stepper(cfg) as st:
        st.set_field(**FIELD)
        st.set_state(psi0)
        st.start(gpe.START_EULER)
        st.step(12)
        got = st.get_state(0)
        st.set_state(psi0)
        st.itp(3, 1e-4)
        relaxed = st.get_state(0)
    a = psi0.copy()
    b = oracle.forward_euler(L, p, a, cfg.dt)
    oracle.leapfrog3(L, p, a, b, cfg.dt, 12, t0=cfg.dt)
    assert rel_l2(got, b) < 1e-13
    ref = psi0 / np.sqrt(oracle.norm(L, p, psi0))
    for _ in range(3):
        nxt = ref - 1e-4 * oracle.apply_h(L, p, ref)
        ref = nxt / np.sqrt(oracle.norm(L, p, nxt))
    assert rel_l2(relaxed, ref) < 1e-13


def test_batched_launch_equals_single_runs():
    members, alone = [], []
    for i, (lat, dims) in enumerate([("bcc", (33, 17, 4)), ("fcc", (12, 10, 3)), ("bcc", (64, 8, 3))]):
        cfg = _run(lat, 3, dims)
        psi0 = random_state(cfg.shape, 20 + i)
        for group in (members, alone):
            st = gpe.Stepper(cfg)
            st.set_field(**FIELD)
            st.set_state(psi0)
            st.start(gpe.START_EULER)
            group.append(st)
    with gpe.Ensemble(members) as ens:
        ens.step(4, graph_sweeps=4)
        ens.step(2)
    for m, s in zip(members, alone):
        s.step(6)
        np.testing.assert_array_equal(m.get_state(0), s.get_state(0))
        m.close()
        s.close()


def test_reverse_sweep_matches_finite_differences():
    cfg = _run("bcc", 3, (13, 10, 3))
    psi0, target = random_state(cfg.shape, 1), random_state(cfg.shape, 2)
    with gpe.Stepper(cfg) as st:
        def value(trap):
            st.set_trap(trap)
            st.set_field(**FIELD)
            st.set_state(psi0)
            return st.adjoint(10, 4, gpe.OBJ_OVERLAP, target)
        res = value((1.0, 1.0, 1.0))
        h = 1e-4  # central differences of a smooth J: O(h^2) against O(eps J / h)
        fd = (value((1.0, 1.0 + h, 1.0))["J"] - value((1.0, 1.0 - h, 1.0))["J"]) / (2 * h)
    assert res["grad_trap"][1] == pytest.approx(fd, rel=1e-5)
