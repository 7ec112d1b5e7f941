"""The traversal tuner on the host stand-in, where the time of a sweep is its number of waves."""
import pytest

from spacetime_amd import gpe
from stand_in import stand_in, started  # noqa: F401


@pytest.mark.parametrize("lat,ncomp,precision,dims,rows", [
    ("fcc", 3, gpe.FP32, (19, 19, 3), 19), ("fcc", 3, gpe.FP64, (17, 17, 4), 17), ("bcc", 3, gpe.FP32, (64, 40, 5), 8)])
def test_no_trials_and_nothing_cached_leaves_the_traversal_alone(stand_in, lat, ncomp, precision, dims, rows):  # noqa: F811
    with started(lat, ncomp, precision, dims) as st:
        before = st.traversal()
        assert before["tile_rows"] == rows
        st.step(1)
        launch = stand_in.sweep()
        t = st.autotune(0)
        assert {k: t[k] for k in before} == before and st.traversal() == before
        st.step(1)
        assert stand_in.sweep() == launch
        st.set_traversal(5, 2, 1)  # a traversal of the caller's own stays too
        st.autotune(0)
        assert st.traversal() == dict(tile_rows=5, xcd_remap=2, x_per_lane=1)


@pytest.mark.parametrize("lat,ncomp,precision,dims", [
    ("fcc", 3, gpe.FP32, (19, 19, 19)), ("a15", 1, gpe.FP32, (9, 11, 9)), ("fcc", 1, gpe.FP32, (35, 31, 35)),
    ("cube", 1, gpe.FP32, (27, 29, 27)), ("bcc", 3, gpe.FP32, (9, 9, 9)), ("fcc", 3, gpe.FP64, (17, 17, 5)),
    ("bcc", 5, gpe.FP64, (21, 21, 3)), ("c15", 5, gpe.FP32, (20, 7, 2)), ("bcc", 3, gpe.FP32, (64, 40, 4))])
def test_tuning_is_never_slower_than_not_tuning(stand_in, lat, ncomp, precision, dims):  # noqa: F811
    with started(lat, ncomp, precision, dims) as st:
        st.step(1)
        untuned = stand_in.sweep()["waves"]
        st.set_traversal(1, 0, 1)  # the candidates do not depend on where the context stands
        t = st.autotune(3)
        st.step(1)
        tuned = stand_in.sweep()["waves"]
        assert tuned <= untuned and t["ms_per_sweep"] == tuned
