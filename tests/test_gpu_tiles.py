"""Tile heights of sweeps that were not tuned: boxes whose lines fill waves only in some heights, with
a remainder of rows in the last tile, one tile for the whole plane and a last tile that leaves whole
waves empty.

Tolerance: a sweep rounds a value a few times at 6e-8 (FP32); 12 steps that add up linearly stay
below 5e-6 of the state's norm.  In FP64 the same count gives 1e-13."""
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


BOXES = [("a15", 1, gpe.FP32, (20, 20, 2)), ("fcc", 3, gpe.FP32, (19, 19, 3)),
         ("c15", 5, gpe.FP32, (18, 18, 2)), ("z", 5, gpe.FP32, (20, 21, 2)),
         ("bcc", 1, gpe.FP32, (50, 50, 2)), ("cube", 1, gpe.FP32, (3, 47, 2)),
         ("cube", 3, gpe.FP32, (96, 10, 3)), ("bcc", 3, gpe.FP32, (5, 3, 4)),
         ("fcc", 1, gpe.FP64, (19, 13, 3)), ("bcc", 5, gpe.FP64, (23, 21, 2))]


@pytest.mark.parametrize("lat,ncomp,precision,dims", BOXES)
def test_untuned_box_against_the_oracle(oracle, lat, ncomp, precision, dims):
    cfg = gpe.Config.centred_box(lat, dims, 0.7, ncomp=ncomp, precision=precision, dt=2e-4, c0=60.0, c1=8.0, c2=3.0,
                                 q=0.1 if ncomp > 1 else 0.0)
    L, p = oracle.lattice(lattice.get(lat)), with_field(oracle_params(oracle, cfg), **FIELD)
    psi0 = random_state(cfg.shape, 5)
    with gpe.Stepper(cfg) as st:
        rows = st.traversal()["tile_rows"]
        assert min(8, dims[1]) <= rows <= min(32, dims[1])
        print(lat, dims, "rows", rows)
        st.set_field(**FIELD)
        st.set_state(psi0)
        st.start(gpe.START_EULER)
        st.step(12)
        got = st.get_state(0)
        st.set_traversal(min(8, dims[1]), st.traversal()["xcd_remap"], st.traversal()["x_per_lane"])
        st.set_state(psi0)
        st.start(gpe.START_EULER)
        st.step(12)
        np.testing.assert_allclose(st.get_state(0), got, rtol=0, atol=5e-6 * np.abs(got).max())
    a = psi0.copy()
    b = oracle.forward_euler(L, p, a, cfg.dt)
    oracle.leapfrog3(L, p, a, b, cfg.dt, 12, t0=cfg.dt)
    assert rel_l2(got, b) < (5e-6 if precision == gpe.FP32 else 1e-13)
