"""Device memory that contexts keep between calls, on the host stand-in: whatever the library
allocates finds room where only an idle workspace is in the way."""
import ctypes

import numpy as np
import pytest

from spacetime_amd import gpe
from stand_in import stand_in, started  # noqa: F401

BOX = ("bcc", 3, gpe.FP32, (8, 6, 5))


def keep_workspace():
    """A context that holds the workspace of an adjoint run."""
    st = started(*BOX)
    st.set_state(np.zeros(st.config.shape, dtype=np.complex128))
    st.adjoint(60, 30, gpe.OBJ_ENERGY)
    return st


def calls():
    """Name -> (what a program has made before, the call that allocates)."""
    def state():
        return started(*BOX)

    def ensemble():
        return gpe.Ensemble([started(*BOX), started(*BOX)])

    def tall():  # its reduction partials grow with tiles of 10 rows (20 rows of waves a plane, 16 before)
        return started("bcc", 1, gpe.FP64, (2, 11, 400))

    zeros = np.zeros(gpe.Config.centred_box(*BOX[:1], BOX[3], 0.7, ncomp=3).shape, dtype=np.complex128)
    return dict(
        create=(lambda: None, lambda _: started(*BOX)),
        set_state=(state, lambda st: st.set_state(zeros)),
        get_state=(state, lambda st: st.get_state(0)),
        weighted_diff=(state, lambda st: st.weighted_diff(zeros)),
        local_fields=(state, lambda st: st.local_fields(0)),
        autotune=(state, lambda st: st.autotune(1)),
        partials=(tall, lambda st: st.set_traversal(10, 1, 1)),
        ensemble_create=(lambda: [started(*BOX)], lambda m: gpe.Ensemble(m)),
        ensemble_step=(ensemble, lambda e: e.step(50)),
        bandwidth=(lambda: None, lambda _: gpe.stream_bandwidth(1 << 20, 1)),
    )


@pytest.mark.parametrize("name", sorted(calls()))
def test_every_allocation_gets_an_idle_workspace_back(stand_in, name):  # noqa: F811
    before, call = calls()[name]
    with keep_workspace():
        held = before()
        stand_in.limits(capacity=stand_in.counts()["used"] + 1)  # full but for the workspace
        call(held)


def test_fields_of_a_long_adjoint_get_another_runs_workspace(stand_in):  # noqa: F811
    """The field records of more sweeps than before, allocated while the call's own workspace is in use."""
    with keep_workspace(), started("cube", 1, gpe.FP32, (2, 2, 2)) as st:
        st.set_state(np.zeros(st.config.shape, dtype=np.complex128))
        used = stand_in.counts()["used"]
        st.adjoint(3000, 2000, gpe.OBJ_ENERGY)
        need = stand_in.counts()["used"] - used
    with keep_workspace(), started("cube", 1, gpe.FP32, (2, 2, 2)) as st:
        st.set_state(np.zeros(st.config.shape, dtype=np.complex128))
        stand_in.limits(capacity=stand_in.counts()["used"] + need - 1)
        st.adjoint(3000, 2000, gpe.OBJ_ENERGY)


def test_a_traversal_without_room_for_its_partials_is_refused_and_changes_nothing(stand_in):  # noqa: F811
    with started("bcc", 1, gpe.FP64, (2, 11, 400)) as st:
        before = st.traversal()
        stand_in.limits(capacity=stand_in.counts()["used"] + 1)
        with pytest.raises(gpe.GpeError, match="ENOMEM"):
            st.set_traversal(10, 1, 1)
        assert st.traversal() == before
        used = stand_in.counts()["used"]
        st.itp(1, 1e-3)  # its partials are still there
        assert stand_in.counts()["used"] == used


def test_a_failed_growth_of_the_field_records_is_not_taken_for_room(stand_in):  # noqa: F811
    with started("cube", 1, gpe.FP32, (2, 2, 2)) as st:
        zeros = np.zeros(st.config.shape, dtype=np.complex128)
        st.set_state(zeros)
        st.adjoint(600, 200, gpe.OBJ_ENERGY)  # workspace made, records for 1024 sweeps
        st.set_state(zeros)
        # room for the larger workspace, none for 4096 records (the old ones are freed first)
        stand_in.limits(max_block=400000)
        with pytest.raises(gpe.GpeError, match="EDEVICE"):
            st.adjoint(3000, 60, gpe.OBJ_ENERGY)
        stand_in.limits()
        st.set_state(zeros)
        st.adjoint(600, 200, gpe.OBJ_ENERGY)


@pytest.mark.parametrize("precision,fp64", [(gpe.FP32, False), (gpe.FP64, False), (gpe.FP32, True)])
def test_buffers_that_fit_only_one_by_one(stand_in, precision, fp64):  # noqa: F811
    """One block of every buffer does not fit (or is larger than an allocation may be), the buffers do:
    the run takes them one by one and gives them back; one byte less and it is refused, with nothing
    left behind."""
    with started("bcc", 3, precision, (8, 6, 5)) as st:
        zeros = np.zeros(st.config.shape, dtype=np.complex128)

        def run():
            st.set_state(zeros)
            return st.adjoint(30, 10, gpe.OBJ_OVERLAP, zeros, fp64)

        whole = run()  # the field records and the copy stream are made
        used = stand_in.counts()["used"]
        stand_in.limits(max_block=400000)  # a level has 69120 or 138240 bytes, staging 138240
        before = stand_in.counts()["allocs"]
        # a larger run than the kept block holds
        st.set_state(zeros)
        r = st.adjoint(40, 10, gpe.OBJ_OVERLAP, zeros, fp64)
        assert stand_in.counts()["allocs"] - before > 20 and r["checkpoint_bytes"] > whole["checkpoint_bytes"]
        assert stand_in.counts()["used"] < used  # not even the old block is kept
        base = stand_in.counts()["used"]
        st.set_state(zeros)
        with pytest.raises(gpe.GpeError, match="ENOMEM"):
            stand_in.limits(capacity=base + 1000000, max_block=400000)
            st.adjoint(40, 10, gpe.OBJ_OVERLAP, zeros, fp64)
        assert stand_in.counts()["used"] == base
        stand_in.limits()
        run()


def test_a_program_can_have_the_workspace_back(stand_in):  # noqa: F811
    with started(*BOX) as st:
        zeros = np.zeros(st.config.shape, dtype=np.complex128)
        st.set_state(zeros)
        st.adjoint(2, 2, gpe.OBJ_ENERGY)  # the field records are made
        st.release_workspace()
        used = stand_in.counts()["used"]
        st.set_state(zeros)
        st.adjoint(30, 10, gpe.OBJ_ENERGY)
        assert stand_in.counts()["used"] > used
        st.release_workspace()
        assert stand_in.counts()["used"] == used
        st.release_workspace()  # nothing to give
        st.set_state(zeros)
        st.adjoint(30, 10, gpe.OBJ_ENERGY)
    assert stand_in.lib.gpe_release_workspace(None) == -22


@pytest.mark.parametrize("nsweeps,every,levels", [(30, 10, 10), (30, 50, 30), (1, 2, 1), (2, 2, 2), (7, 8, 7)])
def test_adjoint_reports_the_levels_of_its_longest_segment(stand_in, nsweeps, every, levels):  # noqa: F811
    with started(*BOX) as st:
        st.set_state(np.zeros(st.config.shape, dtype=np.complex128))
        r = st.adjoint(nsweeps, every, gpe.OBJ_ENERGY)
        level = 8 * 3 * 8 * 6 * 5 * 12  # bytes: FP32 spinors of 8x6x5 cells of 12 (whole lines, no padding)
        assert r["segment_bytes"] == levels * level
        assert r["checkpoint_bytes"] == 2 * -(-nsweeps // every) * level


def test_a_context_is_made_with_few_runtime_calls(stand_in):  # noqa: F811
    """Two levels, one block of tables and results, the partials; one pinned buffer; one copy: an
    ensemble or a parameter study pays for each of them per member."""
    before = stand_in.counts()
    with gpe.Stepper(gpe.Config.centred_box("bcc", (8, 6, 5), 0.7, ncomp=3, precision=gpe.FP64, dt=1e-4)):
        after = stand_in.counts()
    assert {k: after[k] - before[k] for k in ("allocs", "host_allocs", "copies")} == dict(allocs=4, host_allocs=1, copies=1)
    assert stand_in.counts()["used"] == before["used"]
