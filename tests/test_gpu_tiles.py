"""Points-only passes run tile by tile (a quad per thread, rings closed inside
a tile); a full refinement runs the fused and vertex kernels.  Same bytes from
both at the edges of the tiles: levels of just under, exactly and just over
one tile of 256 quads, the change to tiles of 1024, remainders, boundaries,
creases, vertices that are not regular, and points that are not finite."""
import numpy as np
import pytest

from halfedgecatmullclark_amd import cage as C
from tests.helpers import assert_bytes_equal

pytestmark = pytest.mark.gpu

RULES = [("scatter", 0), ("gather", 16), ("plain_scatter", 32), ("plain_gather", 16 | 32)]


def grid(nu, nv):
    """an open sheet of nu x nv quads"""
    i, j = np.meshgrid(np.arange(nu + 1), np.arange(nv + 1), indexing="ij")
    pts = np.stack([i, j, 0.3 * np.sin(i + 2 * j)], -1).reshape(-1, 3).astype(np.float32)
    v = lambda a, b: a * (nv + 1) + b
    faces = [[v(a, b), v(a + 1, b), v(a + 1, b + 1), v(a, b + 1)] for a in range(nu) for b in range(nv)]
    return C.from_faces(pts, faces, creases=[(v(1, b), v(1, b + 1), 1.3) for b in range(nv)] if nu > 1 else [])


# (a level d >= 2 has H0 4^(d-1) quads)
SMALL = [("cube", C.cube(0), 4), ("torus5x3", C.torus(5, 3), 4), ("torus4x4", C.torus(4, 4), 4),
         ("grid1x1", grid(1, 1), 5), ("grid5x3", grid(5, 3), 4), ("irregular", C.irregular(1, seed=3), 4)]


def canonical(p):
    """every NaN alike"""
    return np.where(np.isnan(p), np.float32(np.nan), p)


def tiled(c, D, rule):
    """points of a full refinement, and of two points-only passes after it"""
    import torch
    from halfedgecatmullclark_amd import capi
    st = torch.cuda.current_stream().cuda_stream
    ds = capi.DeviceSubd(c, D)
    ds.refine(15 | rule, st)
    want = ds.download()["points"]
    out = []
    for _ in range(2):
        t = torch.full((ds.n["Vcum"][D], 3), 7.0, device="cuda")
        ds.refine_points(None, t.data_ptr(), rule, st)
        out.append(t.cpu().numpy())
    ds.close()
    return want, out


@pytest.mark.parametrize("rule", [r[1] for r in RULES], ids=[r[0] for r in RULES])
def test_small_tiles(rule):
    import torch
    from halfedgecatmullclark_amd import capi
    for name, c, D in SMALL:
        want, got = tiled(c, D, rule)
        for g in got:
            assert_bytes_equal(g, want, name)
    b = capi.Batch([c for _, c, _ in SMALL], [D for _, _, D in SMALL])
    b.refine(15 | rule)
    want = [b.download(i)["points"].copy() for i in range(len(SMALL))]
    for _ in range(2):
        b.refine_points(None, rule)
        torch.cuda.synchronize()
        for i, (name, _, _) in enumerate(SMALL):
            assert_bytes_equal(b.download(i)["points"], want[i], f"batch {name}")
    b.close()


@pytest.mark.parametrize("rule", [0, 16], ids=["scatter", "gather"])
def test_big_tiles(rule):
    c = C.torus(65, 33)   # 549120 quads at level 4: 536 tiles of 1024 and a remainder
    want, got = tiled(c, 5, rule)
    for g in got:
        assert_bytes_equal(g, want, "torus65x33")


@pytest.mark.parametrize("rule", [r[1] for r in RULES], ids=[r[0] for r in RULES])
def test_points_not_finite(rule):
    c = C.torus(5, 3)
    p = c.vertex_points
    p[1, 0], p[6, 1], p[9, 2], p[12, 0], p[13, 0] = np.inf, np.nan, -0.0, 3e38, -3e38
    want, got = tiled(c, 4, rule)
    for g in got:
        assert_bytes_equal(canonical(g), canonical(want), "not finite")


@pytest.mark.parametrize("name,cage,depth",
                         [("torus4x4_1", C.torus(4, 4), 1), ("torus5x3", C.torus(5, 3), 3), ("torus4x4", C.torus(4, 4), 3),
                          ("grid1x1", grid(1, 1), 5), ("grid5x3", grid(5, 3), 4), ("irregular", C.irregular(1, seed=3), 4),
                          ("torus65x33", C.torus(65, 33), 5)], ids=lambda x: x if isinstance(x, str) else "")
def test_normal_tiles(name, cage, depth):
    """vertex normals of the finest level, the oracle's bytes: one tile and
    part of one, levels of 1024-quad tiles with a remainder (torus65x33),
    boundaries, and vertices that are not regular"""
    import torch
    from halfedgecatmullclark_amd import capi
    from oracle import oracle as O
    st = torch.cuda.current_stream().cuda_stream
    ds = capi.DeviceSubd(cage, depth)
    ds.refine(15, st)
    H = ds.n["H"][depth]
    out = torch.full((H, 3), 7.0, device="cuda")
    ds.halfedge_normals(out.data_ptr(), True, st)
    got = out.cpu().numpy()
    want = O.halfedge_normals(ds.download(), depth, True)
    ds.close()
    assert_bytes_equal(got, np.ascontiguousarray(want).reshape(got.shape), name)


@pytest.mark.parametrize("rule", [r[1] for r in RULES], ids=[r[0] for r in RULES])
def test_two_rings_at_a_vertex(rule):
    """both close inside one tile (level 2: the quads of 16 cage faces)"""
    import torch
    from halfedgecatmullclark_amd import capi
    from tests.helpers import welded_tori
    c, D = welded_tori(3, 3, 0, 4), 4
    want, got = tiled(c, D, rule)
    for g in got:
        assert_bytes_equal(g, want, "welded")
    b = capi.Batch([c, C.torus(4, 4)], [D, 3])
    b.refine(15 | rule)
    want = [b.download(i)["points"].copy() for i in range(2)]
    for _ in range(2):
        b.refine_points(None, rule)
        torch.cuda.synchronize()
        for i in range(2):
            assert_bytes_equal(b.download(i)["points"], want[i], f"batch {i}")
    b.close()


def test_rules_on_two_streams():
    """creased and uncreased passes of one subd, overlapping, each into its
    own buffer: the vertices at sharp edges, which only the creased rules
    leave to the vertex kernel, are written in every pass"""
    import torch
    from halfedgecatmullclark_amd import capi
    c, D = C.torus(24, 16, ring_sharpness=((0, 5.0), (3, 2.5), (8, 4.0))), 6
    ds = capi.DeviceSubd(c, D)
    want = {}
    for rule in (0, 32):
        ds.refine(15 | rule)
        want[rule] = torch.from_numpy(ds.download()["points"]).cuda()
    streams = {rule: torch.cuda.Stream() for rule in want}
    out = {rule: [torch.full((ds.n["Vcum"][D], 3), 7.0, device="cuda") for _ in range(12)] for rule in want}
    torch.cuda.synchronize()
    for k in range(12):
        for rule, s in streams.items():
            ds.refine_points(None, out[rule][k].data_ptr(), rule, s.cuda_stream)
    torch.cuda.synchronize()
    for rule in want:
        for k, t in enumerate(out[rule]):
            assert torch.equal(t.view(torch.int32), want[rule].view(torch.int32)), (rule, k)
    ds.close()


# (level 4 has 256 nu nv quads; the split of a full refinement starts at 655360)
SPLITS = [("below", 59, 43), ("exact", 64, 40), ("above", 61, 42)]


@pytest.mark.parametrize("variant", ["uv", "nouv"])
@pytest.mark.parametrize("name,nu,nv", SPLITS, ids=[s[0] for s in SPLITS])
def test_split_edge(name, nu, nv, variant):
    """full refinements whose largest level has just under, exactly and just
    over the quads from which its points follow its children (649472, 655360
    and 655872: 640 tiles of 1024 and half of one), the oracle's bytes"""
    from halfedgecatmullclark_amd import capi
    from oracle import oracle as O
    c, D = C.torus(nu, nv), 5
    ds = capi.DeviceSubd(c, D, variant)
    b = capi.Batch([c, C.cube(0)], [D, 3], variant)
    ds.set_timing(True)
    for rule, flags in ((0, 0), (16, O.GATHER)):
        want = O.refine(c, D, O.ALL | flags)
        ds.refine(15 | rule)
        ds.synchronize()
        names = [n for n, _ in ds.timings()]
        assert ("level_points" in names) == (name != "below")
        b.refine(15 | rule)
        for got in (ds.download(), b.download(0)):
            assert_bytes_equal(got["points"], want["points"], "points")
            for k in ("twinID", "edgeID", "vertexID"):
                assert np.array_equal(got["halfedges"][k], want["halfedges"][k]), k
    ds.close()
    b.close()


def test_normals_of_two_rings_at_a_vertex():
    """the halfedges of both rings of a shared vertex get their own ring's
    normal"""
    import torch
    from halfedgecatmullclark_amd import capi
    from oracle import oracle as O
    from tests.helpers import welded_tori
    st = torch.cuda.current_stream().cuda_stream
    for c, depth in ((welded_tori(3, 3, 0, 4), 1), (welded_tori(3, 3, 0, 4), 2), (welded_tori(5, 4, 7, 2), 4)):
        ds = capi.DeviceSubd(c, depth)
        ds.refine(15, st)
        out = torch.full((ds.n["H"][depth], 3), 7.0, device="cuda")
        ds.halfedge_normals(out.data_ptr(), True, st)
        got = out.cpu().numpy()
        want = O.halfedge_normals(ds.download(), depth, True)
        ds.close()
        assert_bytes_equal(got, np.ascontiguousarray(want).reshape(got.shape), f"welded {c.H} {depth}")
