"""Launches that sweeps really make, computed without a device: the tile heights of
untuned sweeps and FP64 rows packed into whole waves (decode_rows<1>, lane_coord of gpe_device.h),
emulated on the host's own numbers.  Every wave stays inside the box and the waves cover each unknown
exactly once."""
import ctypes

import numpy as np
import pytest

from spacetime_amd import gpe
from stand_in import stand_in, started  # noqa: F401


def plan(cfg, ty=0, flags=1, xpl=1):
    p = gpe._Plan()
    rc = gpe.load_library().gpe_plan_sweep(cfg.to_c(), ty, flags, xpl, ctypes.byref(p))
    return rc, p


# lanes of the waves that carry values decide: see the counts beside each box
HEIGHTS = [("fcc", 3, gpe.FP32, (19, 19, 3), 19),   # 10 pairs a row: 190 of 192 slots in one tile, 80 of 128 in 8 rows
           ("a15", 1, gpe.FP32, (20, 20, 2), 12),   # 10 pairs: 12 and 8 rows in 2 waves each, 200 of 256 (8 rows: of 384)
           ("bcc", 1, gpe.FP32, (3, 47, 2), 24),    # 2 pairs: tiles of 24 rows in a wave each, 94 of 128 (8 rows: of 384)
           ("cube", 3, gpe.FP32, (96, 10, 3), 10),  # 48 pairs: 480 of 512; tiles of 8 and 2 rows 480 of 768
           ("bcc", 3, gpe.FP32, (5, 3, 4), 3),      # the plane
           ("bcc", 3, gpe.FP32, (128, 128, 8), 8),  # full lines keep 8 rows
           ("fcc", 3, gpe.FP64, (17, 17, 5), 17),   # 289 of 320 lanes; one row a wave 17 of 64
           ("bcc", 3, gpe.FP64, (64, 40, 3), 8),    # full lines
           ("c15", 5, gpe.FP32, (57, 57, 2), 8)]    # taller tiles would leave an XCD's cache


@pytest.mark.parametrize("lat,ncomp,precision,dims,rows", HEIGHTS)
def test_height_of_an_untuned_sweep(stand_in, lat, ncomp, precision, dims, rows):  # noqa: F811
    with started(lat, ncomp, precision, dims) as st:
        rc, p = plan(st.config)
        assert rc == 0 and p.tile_rows == rows == st.traversal()["tile_rows"]
        st.step(1)
        launch = stand_in.sweep()
        assert (p.rows, p.x_per_lane, p.tile_rows, p.waves) == tuple(launch[k] for k in ("rows", "x_per_lane", "tile_rows", "waves"))


PACKED = [("bcc", 5, (70, 11, 4)), ("fcc", 1, (17, 17, 3)), ("fcc", 3, (19, 13, 2)), ("cube", 1, (75, 61, 9)),
          ("cube", 3, (1, 40, 3)), ("bcc", 3, (7, 41, 3)), ("a15", 1, (30, 30, 2)), ("c15", 5, (20, 20, 2)),
          ("z", 3, (5, 9, 3)), ("bcc", 1, (40, 40, 3)), ("bcc", 3, (96, 9, 2)), ("cube", 1, (2, 1, 7))]


@pytest.mark.parametrize("lat,ncomp,dims", PACKED)
def test_packed_fp64_rows_cover_the_box(stand_in, lat, ncomp, dims):  # noqa: F811
    nx, ny, nz = dims
    packed = 0
    with started(lat, ncomp, gpe.FP64, dims) as st:
        for ty in (0, 1, 2, 3, 5, 8, 10, 16, 31, 1024):
            for flags in (0, 1, 2, 3):
                rc, p = plan(st.config, ty, flags, 1)
                assert rc == 0
                if ty:
                    st.set_traversal(ty, flags, 1)
                    st.step(1)
                    launch = stand_in.sweep()
                    assert (p.rows, p.tile_rows, p.waves) == (launch["rows"], launch["tile_rows"], launch["waves"])
                assert p.blocks * 4 >= p.waves and p.tile_rows % p.rows == 0
                if p.rows == 1:
                    continue
                packed += 1
                assert p.pairs == nx and p.rows == p.tile_rows and p.row_groups == 1
                w = np.arange(4 * p.blocks, dtype=np.int64)
                if p.xcd_remap & 2:
                    v, q = w % p.V, w // p.V
                    seg, q = q % p.nseg, q // p.nseg
                else:
                    seg, q = w % p.nseg, w // p.nseg
                    v, q = q % p.V, q // p.V
                z, tile = q % nz, q // nz
                y0 = tile * p.tile_rows
                valid = (w < p.waves) & (seg * 64 < (ny - y0) * nx)
                slot = seg[valid, None] * 64 + np.arange(64)
                v, z, y0 = (a[valid, None] for a in (v, z, y0))
                assert np.all((z >= 0) & (z < nz) & (y0 < ny))
                r, x = slot // nx, slot % nx
                nrow = np.minimum(ny - y0, p.rows)
                live = r < nrow
                assert np.all(y0 + np.minimum(r, nrow - 1) < ny)  # masked lanes read a row of the box
                count = np.zeros((nz, ny, p.V, nx), dtype=np.int32)
                zz, vv, yy = (np.broadcast_to(a, slot.shape) for a in (z, v, y0 + r))
                np.add.at(count, (zz[live], yy[live], vv[live], x[live]), 1)
                assert count.min() == 1 and count.max() == 1, (ty, flags)
    assert packed or lat == "cube"


def test_bad_plans_are_refused():
    cfg = gpe.Config(lattice="bcc", ncomp=3, precision=gpe.FP64, dims=(8, 8, 8))
    assert plan(cfg, 0, 9, 7)[0] == 0  # the untuned launch, whatever else is given
    for bad in ((-1, 1, 1), (1025, 1, 1), (8, 4, 1), (8, 1, 2), (8, 1, 0)):
        assert plan(cfg, *bad)[0] == -22
    assert plan(gpe.Config(lattice="bcc", dims=(0, 8, 8)))[0] == -22


@pytest.mark.parametrize("lat,ncomp,dims,rows", [
    # packed rows were slower than one row a wave here (times of one row's speed)
    ("bcc", 1, (46, 113, 112), 1),   # 0.90: 46 values in lines of 48
    ("fcc", 1, (56, 102, 102), 1),   # 0.92: 7 of 8 lanes full without
    ("cube", 3, (110, 192, 191), 1), # 0.96
    ("cube", 5, (75, 30, 30), 1),    # 0.92: 1800 waves
    ("c15", 5, (200, 11, 10), 1),    # 0.84: 17 MB between the unknowns of a cell
    ("a15", 3, (34, 8, 7), 1),       # 0.93: one tile
    ("z", 5, (34, 13, 13), 1),       # 0.96
    # and faster here
    ("fcc", 5, (40, 81, 81), 8),     # 1.18
    ("bcc", 3, (70, 69, 70), 8),     # 1.24
    ("c15", 1, (70, 27, 27), 8),     # 1.13
    ("cube", 1, (40, 418, 419), 8),  # 1.17
    ("a15", 5, (88, 28, 28), 8),     # 1.05
    ("z", 3, (20, 20, 20), 8)])
def test_rows_are_packed_where_that_was_faster(lat, ncomp, dims, rows):
    cfg = gpe.Config(lattice=lat, ncomp=ncomp, precision=gpe.FP64, dims=dims)
    rc, p = plan(cfg, 8, 1, 1)
    assert rc == 0 and p.rows == rows
