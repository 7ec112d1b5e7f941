"""Generate csrc/lattice_tables.h (C++ constant tables) from the JSON unit-cell tables.

Per lattice: V, max degree, block edges, per-unknown positions and dual volumes, and the
faces padded to the max degree (pad faces: offset 0, target = self, hodge 0) in packed
form (dx+1) | (dy+1) << 2 | (dz+1) << 4 | target << 8.
"""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.dirname(os.path.dirname(HERE)))

from spacetime_amd import lattice  # noqa: E402

OUT = os.path.join(os.path.dirname(HERE), "csrc", "lattice_tables.h")


def _rings(V, near):
    """The unknowns in rings of four, each a same-cell neighbour of the next, or None."""
    used, out = [False] * V, []

    def rest():
        if False not in used:
            return True
        a = used.index(False)
        for b in near[a]:
            for d in near[a]:
                for c in near[b]:
                    ring = (a, b, c, d)
                    if len(set(ring)) < 4 or any(used[q] for q in ring) or c not in near[d]:
                        continue
                    for q in ring:
                        used[q] = True
                    out.extend(ring)
                    if rest():
                        return True
                    del out[-4:]
                    for q in ring:
                        used[q] = False
        return False

    return out if V % 4 == 0 and rest() else None


def device_order(lat):
    """(order, rings): the unknown at each place of the device's numbering of a cell, and whether
    the places are rings of four: a workgroup of the sweep takes four consecutive unknowns, and in a
    ring place p has neighbours at p ^ 1 and p ^ 3 of the same cell.  Lattices without such rings
    keep the table's order."""
    near = []
    for v in range(lat.V):
        fs = range(lat.face_start[v], lat.face_start[v + 1])
        near.append(sorted({int(lat.face_tgt[f]) for f in fs if not lat.face_d[f].any()} - {v}))
    ring = _rings(lat.V, near) if lat.max_degree == 4 else None
    return (ring, 1) if ring else (list(range(lat.V)), 0)


def main():
    lines = ["// Generated by spacetime_amd/tables/gen_header.py from tables/*.json -- do not edit.",
             "// Unit-cell tables of the reference's mesh.h files (see tables/*.json provenance).",
             "#pragma once", "", "namespace gpe {", "",
             "struct LatticeTable {", "    int V, deg;", "    double block_width[3];  // block edges (x, y, z)", "    const double *pos;  // V*3",
             "    const double *vol;  // V", "    const int *face;    // V*deg packed",
             "    const double *hodge; // V*deg (0 for pad faces)",
             "    // the device's numbering of a cell's unknowns: order[p] is the unknown at place p; rings: place",
             "    // p has same-cell neighbours at p ^ 1 and p ^ 3",
             "    const int *order;    // V", "    int rings;", "};", ""]
    names = []
    for name in lattice.LATTICES:
        lat = lattice.get(name)
        deg = lat.max_degree
        packed = []
        hodge = []
        for v in range(lat.V):
            fs, fe = lat.face_start[v], lat.face_start[v + 1]
            for f in range(fs, fe):
                d = lat.face_d[f] + 1
                packed.append(int(d[0] | (d[1] << 2) | (d[2] << 4) | (int(lat.face_tgt[f]) << 8)))
                hodge.append(float(lat.face_hodge[f]))
            for _ in range(deg - (fe - fs)):
                packed.append(int(1 | (1 << 2) | (1 << 4) | (v << 8)))
                hodge.append(0.0)
        fmt = lambda xs: ", ".join(repr(float(x)) for x in xs)  # noqa: E731
        lines.append("static const double %s_pos[] = {%s};" % (name, fmt(lat.pos.reshape(-1))))
        lines.append("static const double %s_vol[] = {%s};" % (name, fmt(lat.vol)))
        lines.append("static const int %s_face[] = {%s};" % (name, ", ".join(str(p) for p in packed)))
        lines.append("static const double %s_hodge[] = {%s};" % (name, fmt(hodge)))
        order, rings = device_order(lat)
        lines.append("static const int %s_order[] = {%s};" % (name, ", ".join(str(v) for v in order)))
        lines.append("")
        names.append("    {%d, %d, {%r, %r, %r}, %s_pos, %s_vol, %s_face, %s_hodge, %s_order, %d}," % (
            lat.V, deg, float(lat.block_dims[0]), float(lat.block_dims[1]), float(lat.block_dims[2]),
            name, name, name, name, name, rings))
    lines.append("static const LatticeTable kLattices[%d] = {" % len(names))
    lines += names
    lines += ["};", "", "}  // namespace gpe", ""]
    with open(OUT, "w") as f:
        f.write("\n".join(lines))
    print("wrote", OUT)


if __name__ == "__main__":
    main()
