"""Reductions whose waves take several chunks each (boxes of more row groups than resident waves), the
norm of more than 65536 workgroups (summed in two stages), and non-finite values wherever they sit,
against the FP64 oracle and direct sums on the stored values.

Tolerance: as for the smaller boxes, 1e-12 relative is 4500 eps, for sums of up to 4.9e6 terms in the
strided and tree order of the kernels (a few hundred eps) of ~50 roundings each; a chunk left out is
1e-4 of them.  Imaginary time in FP64 adds three steps of a few eps a value: 1e-12 as in the small
boxes' 25 steps."""
import numpy as np
import pytest

from helpers import oracle_params, random_state, rel_l2, with_field
from oracle_lib import Oracle
from spacetime_amd import gpe, lattice, states

pytestmark = pytest.mark.gpu

FIELD = dict(bq=4e-3, bb=(0.01, -0.02, 0.05), bq_quad=2e-3, bb_quad=(0.05, 0.02, -0.03))


@pytest.fixture(scope="module")
def oracle():
    return Oracle()


def config(lat, ncomp, precision, dims, **kw):
    return gpe.Config.centred_box(lat, dims, 0.7, ncomp=ncomp, precision=precision, dt=1e-4, c0=60.0, c1=8.0, c2=3.0,
                                  q=0.1 if ncomp > 1 else 0.0, trap=(1.0, 1.1, 0.05), trap_offset=0.5,
                                  center=(0.1, 0.0, -0.2), **kw)


def spin_density(psi):
    """psi^dag f psi and the reference's local spin (x, y of the spinor over sqrt(n), z undivided)."""
    C = psi.shape[0]
    n = np.sum(np.abs(psi) ** 2, axis=0)
    if C == 1:
        return n, np.zeros(n.shape + (3,)), np.zeros(n.shape + (3,))
    F = (C - 1) // 2
    m = np.arange(F, -F - 1, -1)
    up = sum(np.sqrt(F * (F + 1) - m[i + 1] * (m[i + 1] + 1)) * psi[i].conj() * psi[i + 1] for i in range(C - 1))
    full = np.stack([up.real, up.imag, sum(m[i] * np.abs(psi[i]) ** 2 for i in range(C))], axis=-1)
    o = F - 1
    t = np.sqrt(2.0) * (psi[o].conj() * psi[o + 1] + psi[o + 1].conj() * psi[o + 2])
    with np.errstate(invalid="ignore", divide="ignore"):
        t = np.where(n > 0, t / n, 0.0)
    return n, full, np.stack([t.real, t.imag, np.abs(psi[o]) ** 2 - np.abs(psi[o + 2]) ** 2], axis=-1)


@pytest.mark.parametrize("lat,ncomp,precision,dims", [
    ("bcc", 3, gpe.FP32, (5, 8, 1500)), ("bcc", 1, gpe.FP64, (5, 8, 1500)), ("fcc", 5, gpe.FP64, (3, 9, 800)),
    ("a15", 3, gpe.FP32, (4, 7, 400)),
    ("cube", 1, gpe.FP32, (60, 9, 9000)), ("bcc", 3, gpe.FP32, (20, 8, 800))])
def test_observables_of_waves_with_several_chunks(oracle, lat, ncomp, precision, dims):
    cfg = config(lat, ncomp, precision, dims)
    L = oracle.lattice(lattice.get(lat))
    p = with_field(oracle_params(oracle, cfg), **FIELD)
    with gpe.Stepper(cfg) as st:
        st.set_field(**FIELD)
        st.set_state(random_state(cfg.shape, 5))
        o = st.observables(0)
        psi = st.get_state(0)
    tol = 1e-12
    dv, r = states.dual_volumes(cfg), states.positions(cfg)
    n, F, ref = spin_density(psi)
    assert o.finite
    assert o.norm == pytest.approx(oracle.norm(L, p, psi), rel=tol)
    assert o.energy == pytest.approx(oracle.energy(L, p, psi), rel=tol)
    assert o.expect_h == pytest.approx(oracle.expect_h(L, p, psi), rel=tol)
    assert o.max_density == pytest.approx(n.max(), rel=1e-14)
    np.testing.assert_allclose(o.magnetization, oracle.magnetization(L, p, psi), rtol=tol, atol=tol * o.norm)
    np.testing.assert_allclose(o.moment, np.sum((n * dv)[..., None] * r, axis=(0, 1, 2, 3)), rtol=tol,
                               atol=tol * np.sum(n * dv * np.linalg.norm(r, axis=-1)))
    assert o.spin == pytest.approx(np.sum(np.linalg.norm(F, axis=-1) * dv), rel=tol, abs=1e-14)
    assert o.ref_spin == pytest.approx(np.sum(n * np.linalg.norm(ref, axis=-1) * dv), rel=tol, abs=1e-14)
    assert o.ref_magnetization_z == pytest.approx(np.sum(n * ref[..., 2] * dv), rel=tol, abs=tol * np.sum(n * n * dv))


@pytest.mark.parametrize("lat,ncomp,precision,dims,traversal", [
    ("bcc", 1, gpe.FP64, (2, 150, 150), (1, 1, 1)),   # 67500 workgroups of a sweep: two stages
    ("bcc", 3, gpe.FP64, (2, 148, 148), (1, 1, 1)),   # 65712
    ("bcc", 1, gpe.FP64, (2, 148, 147), (1, 1, 1)),   # 65268: one
    ("bcc", 1, gpe.FP64, (5, 8, 1500), None)])        # several chunks a wave in the norm of the start
def test_imaginary_time_norms_of_many_workgroups(oracle, lat, ncomp, precision, dims, traversal):
    cfg = config(lat, ncomp, precision, dims)
    L, p = oracle.lattice(lattice.get(lat)), oracle_params(oracle, cfg)
    psi = random_state(cfg.shape, 8)
    ref = psi.copy()
    oracle.normalize(L, p, ref)
    for _ in range(3):
        oracle.itp_step(L, p, ref, 1e-4)
    with gpe.Stepper(cfg) as st:
        if traversal:
            st.set_traversal(*traversal)
        st.set_state(psi)
        st.itp(3, 1e-4)
        got = st.get_state(0)
        norm = st.observables(0).norm
    assert norm == pytest.approx(1.0, rel=1e-12)
    assert rel_l2(got, ref) < 1e-12


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 1j * np.inf])
@pytest.mark.parametrize("lat,ncomp,precision,dims", [
    ("bcc", 3, gpe.FP32, (5, 8, 1500)), ("cube", 1, gpe.FP64, (7, 9, 3)), ("fcc", 5, gpe.FP64, (3, 9, 5)),
    ("a15", 1, gpe.FP32, (9, 11, 2))])
def test_a_non_finite_value_is_seen_wherever_it_sits(lat, ncomp, precision, dims, value):
    cfg = config(lat, ncomp, precision, dims)
    nx, ny, nz = dims
    V = cfg.V
    psi = random_state(cfg.shape, 3)
    with gpe.Stepper(cfg) as st:
        for c, z, y, x, v in [(0, 0, 0, 0, 0), (ncomp - 1, nz - 1, ny - 1, nx - 1, V - 1), (ncomp // 2, nz // 2, ny // 2, nx - 1, V // 2),
                              (0, nz - 1, 0, nx // 2, 0), (ncomp - 1, nz // 3, ny - 1, 0, V - 1)]:
            bad = psi.copy()
            bad[c, z, y, x, v] = value
            st.set_state(bad)
            assert not st.observables(0, check=False).finite
            with pytest.raises(gpe.GpeError, match="ERANGE"):
                st.observables(0)
            st.set_state(psi)
            assert st.observables(0).finite
