"""The device's numbering of a cell's unknowns (tables/gen_header.py device_order): a permutation, and
where it claims rings, places 4k..4k+3 form a ring of same-cell neighbours."""
import pytest

from spacetime_amd import lattice
from spacetime_amd.tables.gen_header import device_order


@pytest.mark.parametrize("name", lattice.LATTICES)
def test_device_order(name):
    lat = lattice.get(name)
    order, rings = device_order(lat)
    assert sorted(order) == list(range(lat.V))
    assert rings == (name == "bcc")
    if not rings:
        assert order == list(range(lat.V))
        return
    near = {(int(lat.face_src[f]), int(lat.face_tgt[f])) for f in range(lat.nfaces) if not lat.face_d[f].any()}
    for p in range(lat.V):
        for q in (p ^ 1, p ^ 3):
            assert (order[p], order[q]) in near
