"""Cages that the rare-vertex table does not take (a fan of more than 64
entries) under the tile kernel: every level lists its rare vertices afresh.
Points-only passes, twice, and a full refinement of a level large enough for
its points to follow its children, alone and in a batch, bytes equal to the
oracle's."""
import numpy as np
import pytest

from halfedgecatmullclark_amd import cage as C
from oracle import oracle as O
from tests.helpers import assert_bytes_equal
from tests.test_gpu_rare import RULES, bipyramid, cone, prism, ring_points

pytestmark = pytest.mark.gpu

DEPTH = 4


def drum(k, m):
    """m rings of k quads between two faces of k corners"""
    pts = np.concatenate([ring_points(k, z / m) for z in range(m + 1)]).astype(np.float32)
    faces = [list(range(k))[::-1], [m * k + i for i in range(k)]]
    faces += [[j * k + i, j * k + (i + 1) % k, (j + 1) * k + (i + 1) % k, (j + 1) * k + i]
              for j in range(m) for i in range(k)]
    return C.from_faces(pts, faces, creases=[(0, 1, 2.0), (k, k + 1, 0.8)])


def moved(c, s):
    p = (c.vertex_points + np.float32(0.05) * np.sin(np.float32(7 + s) * c.vertex_points[:, ::-1])).astype(np.float32)
    return np.ascontiguousarray(p)


def with_points(c, p):
    q = c.copy()
    q.vertex_points = p
    return q


CAGES = [("cone65", cone(65)), ("bipyramid65", bipyramid(65)), ("prism65", prism(65)), ("prism9", prism(9))]


@pytest.mark.parametrize("rule,steps,flags", RULES, ids=[r[0] for r in RULES])
def test_points_only(rule, steps, flags):
    import torch
    from halfedgecatmullclark_amd import capi
    st = torch.cuda.current_stream().cuda_stream
    points = [[moved(c, s) for _, c in CAGES] for s in range(2)]
    want = [[O.refine(with_points(c, p), DEPTH, flags)["points"] for (_, c), p in zip(CAGES, ps)] for ps in points]
    for i, (name, c) in enumerate(CAGES):
        for variant in ("uv", "nouv"):
            ds = capi.DeviceSubd(c, DEPTH, variant)
            ds.refine(steps, st)
            for s in range(2):
                p = torch.from_numpy(points[s][i]).cuda()
                out = torch.full((ds.n["Vcum"][DEPTH], 3), 7.0, device="cuda")
                ds.refine_points(p.data_ptr(), out.data_ptr(), steps & 48, st)
                assert_bytes_equal(out.cpu().numpy(), want[s][i], f"{variant} {name}")
            ds.close()
    b = capi.Batch([c for _, c in CAGES], [DEPTH] * len(CAGES))
    b.refine(steps, st)
    for s in range(2):
        p = torch.from_numpy(np.concatenate(points[s])).cuda()
        b.refine_points(p.data_ptr(), steps & 48, st)
        torch.cuda.synchronize()
        for i, (name, _) in enumerate(CAGES):
            assert_bytes_equal(b.download(i)["points"], want[s][i], f"batch {name}")
    b.close()


@pytest.mark.parametrize("rule,steps,flags", RULES[:2], ids=[r[0] for r in RULES[:2]])
def test_large_level(rule, steps, flags):
    """657280 quads at level 4: 641 tiles of 1024 and a remainder"""
    from halfedgecatmullclark_amd import capi
    c = drum(65, 39)
    want = O.refine(c, 5, flags)
    ds = capi.DeviceSubd(c, 5)
    ds.refine(steps)
    got = ds.download()
    ds.close()
    b = capi.Batch([c, prism(9)], [5, 3])
    b.refine(steps)
    bat = b.download(0)
    b.close()
    for k in ("halfedges", "creases", "points"):
        assert_bytes_equal(got[k], want[k], k)
        assert_bytes_equal(bat[k], want[k], f"batch {k}")
