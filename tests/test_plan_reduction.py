"""The chunks of a reduction (reduce_geometry on the host, decode_reduce of gpe_kernels.hip), emulated on
the arguments of the host's own launches: every wave stays inside the box, the waves cover each unknown
exactly once, and there are no more of them than stated."""
import numpy as np
import pytest

from spacetime_amd import gpe
from stand_in import stand_in, started  # noqa: F401


REDUCED = [("cube", 1, (1, 1, 1)), ("cube", 1, (65, 9, 3)), ("cube", 3, (300, 33, 5)), ("bcc", 3, (7, 41, 3)),
           ("bcc", 1, (128, 17, 9)), ("a15", 5, (19, 9, 2)), ("c15", 3, (57, 11, 3)), ("fcc", 3, (177, 11, 2)),
           ("bcc", 3, (5, 8, 1500)), ("z", 1, (3, 2, 90)), ("cube", 1, (700, 70, 2))]


@pytest.mark.parametrize("resident", [8, 768, 1024, 2048])
@pytest.mark.parametrize("lat,ncomp,dims", REDUCED)
def test_chunks_of_a_reduction_cover_the_box(stand_in, lat, ncomp, dims, resident):  # noqa: F811
    nx, ny, nz = dims
    stand_in.lib.stand_in_resident(resident)
    try:
        with started(lat, ncomp, gpe.FP32, dims) as st:
            st.observables(0, check=False)
    finally:
        stand_in.lib.stand_in_resident(1024)
    g = stand_in.reduction()
    V, each = g["V"], g["blocks"] // 8
    groups = g["ntile"] * nz * V
    assert g["blocks"] % 8 == 0 and g["blocks"] <= 2048
    assert g["waves"] <= max(groups, 4 * resident)
    b, wid = np.meshgrid(np.arange(g["blocks"]), np.arange(4), indexing="ij")
    first = ((b & 7) * each * g["per"] + (b >> 3)) * 4 + wid
    count = np.zeros((nz, ny, V, nx), dtype=np.int32)
    for j in range(g["per"]):
        w = (first + 4 * each * j).ravel()
        w = w[w < g["waves"]]  # a wave ends at its first one past the traversal, and they grow with j
        chunk, q = w % g["nseg"], w // g["nseg"]
        v, q = q % V, q // V
        z, y0 = q % nz, q // nz * g["ty"]
        assert np.all(y0 < ny)
        slots = np.minimum(ny - y0, g["rows"]) * nx
        lo = chunk * g["segs"] * 64
        for k in range(64 * g["segs"]):
            p = lo + k
            live = p < np.minimum(lo + 64 * g["segs"], slots)
            np.add.at(count, (z[live], y0[live] + p[live] // nx, v[live], p[live] % nx), 1)
    assert count.min() == 1 and count.max() == 1


def test_reductions_of_large_boxes_take_several_chunks_a_wave(stand_in):  # noqa: F811
    """That the box above really has them at the resident workgroups of the device (1024 and 2048)."""
    for resident, per in ((1024, 5), (2048, 3)):
        stand_in.lib.stand_in_resident(resident)
        with started("bcc", 3, gpe.FP32, (5, 8, 1500)) as st:
            st.observables(0, check=False)
        assert stand_in.reduction()["per"] == per
    stand_in.lib.stand_in_resident(1024)
