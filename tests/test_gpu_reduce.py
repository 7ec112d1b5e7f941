"""Observables over boxes at the edges of their traversal (row groups of 64-slot segments, chunks,
XCD ranges): single unknown rows, lines just over a segment, tiles with a remainder of rows, boxes
with fewer groups than waves, against the FP64 oracle on the stored values.

Tolerance: a sum of N <= 1e6 terms of one sign rounds by at most N eps = 2e-10 and, in the
butterfly and strided order of the kernel, by a few hundred eps; the energy's terms carry ~50
roundings each and cancel by less than 10 here.  1e-12 relative is 4500 eps."""
import numpy as np
import pytest

from helpers import oracle_params, random_state, with_field
from oracle_lib import Oracle
from spacetime_amd import gpe, lattice

pytestmark = pytest.mark.gpu

FIELD = dict(bq=4e-3, bb=(0.01, -0.02, 0.05), bq_quad=2e-3, bb_quad=(0.05, 0.02, -0.03))


@pytest.fixture(scope="module")
def oracle():
    return Oracle()


@pytest.mark.parametrize("lat,ncomp,precision,dims", [
    ("cube", 1, gpe.FP32, (1, 1, 1)), ("cube", 1, gpe.FP64, (65, 9, 3)), ("cube", 3, gpe.FP32, (300, 33, 5)),
    ("bcc", 3, gpe.FP32, (64, 8, 2)), ("bcc", 3, gpe.FP64, (7, 41, 3)), ("bcc", 1, gpe.FP32, (128, 17, 9)),
    ("fcc", 5, gpe.FP32, (33, 10, 4)), ("fcc", 3, gpe.FP64, (2, 3, 20)), ("a15", 5, gpe.FP64, (19, 9, 2)),
    ("c15", 3, gpe.FP32, (29, 12, 3)), ("z", 1, gpe.FP64, (34, 7, 3)),
])
def test_observables_at_traversal_edges(oracle, lat, ncomp, precision, dims):
    cfg = gpe.Config.centred_box(lat, dims, 0.7, ncomp=ncomp, precision=precision, dt=1e-4, c0=60.0, c1=8.0,
                                 c2=3.0, q=0.1, trap=(1.0, 1.1, 1.25), trap_offset=0.5, center=(0.1, 0.0, -0.2))
    L = oracle.lattice(lattice.get(lat))
    p = with_field(oracle_params(oracle, cfg), **FIELD)
    with gpe.Stepper(cfg) as st:
        st.set_field(**FIELD)
        st.set_state(random_state(cfg.shape, 5))
        o = st.observables(0)
        again = st.observables(0)
        psi = st.get_state(0)
    tol = 1e-12
    assert o.finite and o.norm == again.norm and o.energy == again.energy  # a fixed order of summation
    assert o.norm == pytest.approx(oracle.norm(L, p, psi), rel=tol)
    assert o.energy == pytest.approx(oracle.energy(L, p, psi), rel=tol)
    assert o.expect_h == pytest.approx(oracle.expect_h(L, p, psi), rel=tol)
    np.testing.assert_allclose(o.magnetization, oracle.magnetization(L, p, psi), rtol=tol, atol=tol * o.norm)
    assert o.max_density == pytest.approx(np.max(np.sum(np.abs(psi) ** 2, axis=0)), rel=1e-14)
