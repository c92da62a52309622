"""The wavefront-wide solid test where its shortcut must not answer: triangles
whose planes hold nodes or rays, rays through vertices and along edges (a body
aligned with the grid and centred on it), a body far from the origin, small and
ragged boxes, a body much larger and much smaller than the box; geometries in
small units (spacing 1e-3 to 1e-6) and normals that are not unit vectors, where
the absolute tolerances of the crossing test (1.24e-16 on volumes, 1e-14 on a
plane through the node) decide many candidates.  The table, the solid count and
the tie count equal the CPU restatement's exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FACES = [-101, -10, -10, -201, -10, -10]


def box_tris(lo, hi):
    """Twelve triangles of an axis-aligned box, outward normals."""
    c = np.array([[lo[0] if not i & 1 else hi[0], lo[1] if not i & 2 else hi[1],
                   lo[2] if not i & 4 else hi[2]] for i in range(8)], float)
    quads = [(0, 2, 6, 4), (1, 5, 7, 3), (0, 4, 5, 1), (2, 3, 7, 6), (0, 1, 3, 2), (4, 6, 7, 5)]
    return np.array([[*c[a], *c[b], *c[d]] for q in quads for a, b, d in
                     ((q[0], q[1], q[2]), (q[0], q[2], q[3]))])


def octahedron(centre, r, level):
    v = np.array([(1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)], float)
    t = [(v[a], v[b], v[c]) for a in (0, 1) for b in (2, 3) for c in (4, 5)]
    for _ in range(level):
        t = [u for p, q, s in t for m in [[x / np.linalg.norm(x) for x in (p + q, q + s, s + p)]]
             for u in ((p, m[0], m[2]), (q, m[1], m[0]), (s, m[2], m[1]), tuple(m))]
    return np.array([np.concatenate([r * p + centre for p in u]) for u in t])


def normals(tri, centre):
    p = tri.reshape(-1, 3, 3)
    n = np.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0])
    n /= np.linalg.norm(n, axis=1, keepdims=True)
    out = ((p.mean(axis=1) - centre) * n).sum(axis=1) < 0
    n[out] *= -1
    return n


CASES = {
    "grid-aligned box": ((20, 17, 13), (0, 0, 0), 1.0, box_tris((5, 4, 3), (11, 9, 8)), (8, 6.5, 5.5)),
    "box on half nodes": ((20, 17, 13), (0, 0, 0), 1.0, box_tris((5.5, 4.5, 3.5), (11.5, 9.5, 8.5)),
                          (8.5, 7, 6)),
    "octahedron at the centre": ((21, 21, 21), (0, 0, 0), 1.0, octahedron((10, 10, 10), 6.0, 0),
                                 (10, 10, 10)),
    "sphere at the centre": ((21, 21, 21), (0, 0, 0), 1.0, octahedron((10, 10, 10), 6.3, 3),
                             (10, 10, 10)),
    "sphere off the nodes": ((37, 19, 23), (0, 0, 0), 1.0, octahedron((11.17, 9.41, 10.83), 5.7, 4),
                             (11.17, 9.41, 10.83)),
    "far from the origin": ((24, 18, 16), (4e3, -7e3, 2e3), 0.25,
                            octahedron((4003.1, -6997.8, 2002.1), 1.31, 3), (4003.1, -6997.8, 2002.1)),
    "larger than the box": ((9, 8, 7), (0, 0, 0), 1.0, octahedron((4.3, 3.9, 3.2), 40.0, 3),
                            (4.3, 3.9, 3.2)),
    "smaller than a cell": ((9, 8, 7), (0, 0, 0), 1.0, octahedron((4.0, 4.0, 3.0), 0.4, 1),
                            (4.0, 4.0, 3.0)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_table_equals_cpu(pkg, orc, name):
    shape, origin, dx, tri, centre = CASES[name]
    compare(pkg, orc, name, shape, origin, dx, tri, normals(tri, np.array(centre)))


@pytest.mark.parametrize("dx", [1e-3, 1e-4, 3e-5, 1e-5, 1e-6])
@pytest.mark.parametrize("name", ["sphere off the nodes", "box on half nodes", "sphere of many triangles"])
def test_small_units_equal_cpu(pkg, orc, name, dx):
    if name in CASES:
        shape, _, _, tri, centre = CASES[name]
    else:
        shape, centre = (48, 40, 32), (23.31, 19.47, 15.82)
        tri = octahedron(np.array(centre), 9.0, 5)
    nrm = normals(tri, np.array(centre))
    compare(pkg, orc, f"{name}, dx {dx}", shape, (0, 0, 0), dx, tri * dx, nrm)


@pytest.mark.parametrize("length", [1e-12, 1e-8, 1e6])
def test_normals_of_any_length_equal_cpu(pkg, orc, length):
    shape, origin, dx, tri, centre = CASES["sphere off the nodes"]
    compare(pkg, orc, f"normals of length {length}", shape, origin, dx, tri,
            length * normals(tri, np.array(centre)))


def compare(pkg, orc, name, shape, origin, dx, tri, nrm):
    s = pkg.Solver(precision="fp32s", nu=0.01)
    s.define_level(0, shape, periodic=(0, 0, 0))
    s.set_faces(0, FACES)
    n_solid, n_tie = s.build_links(0, tri, nrm, origin=origin, dx=dx)
    want, solid_o, tie_o = orc.build_links27(shape, FACES, tri, nrm, dx=dx, origin=origin)
    print(f"{name}: solid {n_solid}, ties {n_tie}")
    assert np.array_equal(s.download_links(0), np.asarray(want).reshape(27, -1))
    assert n_solid == solid_o and n_tie == tie_o
