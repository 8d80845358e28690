"""Vertices that take their rings from the rare-vertex table, at the sizes
where its lane groups change (4, 8 and 64 entries, a boundary fan having one
entry more than halfedges) and past the largest, where the rare list takes
over: cones (open), bipyramids and prisms, bytes equal to the oracle's for
every rule, alone and in a batch, with both record sizes."""
import numpy as np
import pytest

from halfedgecatmullclark_amd import cage as C
from oracle import oracle as O
from tests.helpers import assert_bytes_equal

pytestmark = pytest.mark.gpu

RULES = [("scatter", 15, O.ALL), ("gather", 15 | 16, O.ALL | O.GATHER), ("plain_scatter", 15 | 32, O.ALL | O.NOCREASES),
         ("plain_gather", 15 | 16 | 32, O.ALL | O.GATHER | O.NOCREASES)]
DEPTH = 3


def ring_points(k, z):
    a = 2 * np.pi * np.arange(k) / k
    return np.stack([np.cos(a), np.sin(a) + 0.1 * np.cos(3 * a), z + 0.05 * np.sin(5 * a)], 1)


def cone(k):
    """k triangles around an apex, open below: a boundary loop of k edges"""
    pts = np.concatenate([[[0.1, 0, 1]], ring_points(k, 0)]).astype(np.float32)
    return C.from_faces(pts, [[0, 1 + i, 1 + (i + 1) % k] for i in range(k)],
                        creases=[(0, 1, 1.5), (0, 2, 0.7), (0, 3, 2.5)][: k % 4])


def fan(k):
    """k triangles around an apex on the boundary: an open fan"""
    a = np.pi * np.arange(k + 1) / k
    pts = np.concatenate([[[0, 0, 0.3]], np.stack([np.cos(a), np.sin(a), 0.2 * np.cos(3 * a)], 1)]).astype(np.float32)
    return C.from_faces(pts, [[0, 1 + i, 2 + i] for i in range(k)], creases=[(0, 2, 1.2)] if k > 1 else [],
                        sharpen_boundaries=k % 2 == 0)


def bipyramid(k):
    pts = np.concatenate([[[0.1, 0, 1]], ring_points(k, 0), [[0, 0.2, -1]]]).astype(np.float32)
    faces = [[0, 1 + i, 1 + (i + 1) % k] for i in range(k)] + [[k + 1, 1 + (i + 1) % k, 1 + i] for i in range(k)]
    return C.from_faces(pts, faces, creases=[(1, 2, 3.0), (2, 3, 0.4), (0, 1, 1.1), (0, 3, 0.9)])


def prism(k):
    """two faces of k corners and k quads"""
    pts = np.concatenate([ring_points(k, 0), ring_points(k, 1)]).astype(np.float32)
    faces = [list(range(k))[::-1], [k + i for i in range(k)]] + [[i, (i + 1) % k, k + (i + 1) % k, k + i]
                                                                 for i in range(k)]
    return C.from_faces(pts, faces, creases=[(0, 1, 2.0), (1, 2, 0.8)])


CAGES = [(f"{f.__name__}{k}", f(k)) for f, ks in ((cone, (3, 4, 5, 8, 9, 64, 65)), (fan, (1, 2, 3, 4, 7, 8, 63, 64)),
                                                   (bipyramid, (3, 5, 8, 9, 64, 65)), (prism, (3, 5, 8, 9, 64, 65)))
         for k in ks]


def check(got, want, what):
    assert_bytes_equal(got["halfedges"], want["halfedges"], f"{what} halfedges")
    assert_bytes_equal(got["creases"], want["creases"], f"{what} creases")
    assert_bytes_equal(got["points"], want["points"], f"{what} points")


@pytest.mark.parametrize("rule,steps,flags", RULES, ids=[r[0] for r in RULES])
def test_rare_vertices(rule, steps, flags):
    from halfedgecatmullclark_amd import capi
    want = [O.refine(c, DEPTH, flags) for _, c in CAGES]
    b = capi.Batch([c for _, c in CAGES], [DEPTH] * len(CAGES))
    b.refine(steps)
    b.refine(steps)   # the captured graph
    for i, (name, c) in enumerate(CAGES):
        check(b.download(i), want[i], f"batch {name}")
        ds = capi.DeviceSubd(c, DEPTH)
        ds.refine(steps)
        check(ds.download(), want[i], name)
        ds.close()
        nd = capi.DeviceSubd(c, DEPTH, variant="nouv")
        nd.refine(steps)
        assert_bytes_equal(nd.download()["points"], want[i]["points"], f"nouv {name} points")
        nd.close()
    b.close()
