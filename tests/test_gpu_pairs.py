"""Cages whose edges the reference's maps do not represent by the larger
halfedge on every level: faces that use an edge twice, and halfedges numbered
at random.  Every point has one owner: the scatter rules give the oracle's
bytes, a points-only pass and a batch the same, and the adjoint is the
transpose.  (The gather rules start from the representative, which in the
reference belongs to a neighbouring edge there; they are not compared.)"""
import numpy as np
import pytest

from halfedgecatmullclark_amd import cage as C
from oracle import oracle as O
from tests.helpers import assert_bytes_equal, permuted, tip_cages
from tests.test_gpu_rare import cone, prism

pytestmark = pytest.mark.gpu

CAGES = tip_cages() + [(f"permuted_{n}", permuted(c, i)) for i, (n, c) in enumerate(
    [("torus", C.torus(5, 4)), ("irregular", C.irregular(1, seed=3)), ("cone5", cone(5)), ("prism65", prism(65))]
    + tip_cages()[3:])]


@pytest.mark.parametrize("depth", [3, 5])
@pytest.mark.parametrize("rule,flags", [(0, 0), (32, O.NOCREASES)], ids=["creased", "plain"])
def test_scatter_points(rule, flags, depth):
    import torch
    from halfedgecatmullclark_amd import capi
    want = [O.refine(c, depth, O.ALL | flags) for _, c in CAGES]
    for (name, c), w in zip(CAGES, want):
        for variant in ("uv", "nouv"):
            ds = capi.DeviceSubd(c, depth, variant)
            ds.refine(15 | rule)
            got = ds.download()
            assert_bytes_equal(got["points"], w["points"], f"{variant} {name}")
            assert_bytes_equal(got["creases"], w["creases"], f"{variant} {name} creases")
            for _ in range(2):
                out = torch.full((ds.n["Vcum"][depth], 3), 7.0, device="cuda")
                ds.refine_points(None, out.data_ptr(), rule, torch.cuda.current_stream().cuda_stream)
                assert_bytes_equal(out.cpu().numpy(), w["points"], f"{variant} {name} points only")
            ds.close()
    b = capi.Batch([c for _, c in CAGES], [depth] * len(CAGES))
    b.refine(15 | rule)
    for k in range(2):
        for i, (name, _) in enumerate(CAGES):
            assert_bytes_equal(b.download(i)["points"], want[i]["points"], f"batch {name} {k}")
        b.refine_points(None, rule)
        b.synchronize()
    b.close()


@pytest.mark.parametrize("name,cage", CAGES, ids=[c[0] for c in CAGES])
def test_adjoint(name, cage):
    import torch
    from halfedgecatmullclark_amd import capi
    depth, rng = 4, np.random.default_rng(5)
    c = cage.copy()
    c.vertex_points = rng.normal(size=(c.V, 3))
    y = O.level(O.refine(c, depth, O.ALL, real=np.float64), "points", depth)
    g = rng.normal(size=y.shape)
    ds = capi.DeviceSubd(cage, depth)
    ds.refine()
    gt, out = torch.from_numpy(g).cuda(), torch.zeros((c.V, 3), dtype=torch.float64, device="cuda")
    ds.refine_points_adjoint(gt.data_ptr(), out.data_ptr(), capi.FP64, torch.cuda.current_stream().cuda_stream)
    # sums of a few thousand products, each of rounding error 2^-53 or less
    assert abs((c.vertex_points * out.cpu().numpy()).sum() - (y * g).sum()) <= 1e-12 * np.abs(y * g).sum()
    ds.close()
