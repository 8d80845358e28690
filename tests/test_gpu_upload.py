"""The cage's way to the device on both sides of its rules: packed or array by
array, lists by one thread or two, with a rare-vertex table or with the list
for one call.  Host refinements of one subd, the cage's points moved and an
adjoint between them, against the oracle and the device-resident adjoint."""
import numpy as np
import pytest

from halfedgecatmullclark_amd import cage as C
from oracle import oracle as O
from tests.helpers import assert_bytes_equal

pytestmark = pytest.mark.gpu

# (arrays from 1 MiB on go one by one, lists by two threads from 32768
# halfedges on, 5000 table entries a level for one call)
CASES = [("irregular3_d3", C.irregular(3), 3),    # packed, one thread, table
         ("irregular4_d2", C.irregular(4), 2),    # packed, one thread, list
         ("irregular5_d2", C.irregular(5), 2),    # by array, two threads, list
         ("torus96x85_d2", C.torus(96, 85), 2),   # by array, one thread, table (empty)
         ("torus128x66_d1", C.torus(128, 66), 1)]  # by array, two threads, neither


@pytest.mark.parametrize("name,cage,depth", CASES, ids=[c[0] for c in CASES])
def test_host_calls_of_one_subd(name, cage, depth):
    import torch
    from halfedgecatmullclark_amd import capi
    c = cage.contiguous()
    s = capi.HostSubd(c, depth)

    def check(flags):
        want = O.refine(c, depth, flags)
        got = s.arrays()
        for k in ("halfedges", "creases", "points"):
            assert_bytes_equal(got[k], want[k], f"{name} {k}")

    s.run("ccs_Refine_Scatter")
    check(O.ALL)
    c.vertex_points *= np.float32(1.25)
    s.run("ccs_Refine_Gather")
    check(O.ALL | O.GATHER)
    g = np.random.default_rng(3).normal(size=(s.n["V"][depth], 3)).astype(np.float32)
    got = s.adjoint(g)
    ds = capi.DeviceSubd(c, depth)
    ds.refine()
    gf, gc = torch.from_numpy(g).cuda(), torch.zeros((c.V, 3), device="cuda")
    ds.refine_points_adjoint(gf.data_ptr(), gc.data_ptr(), 0, torch.cuda.current_stream().cuda_stream)
    assert_bytes_equal(got, gc.cpu().numpy(), f"{name} adjoint")
    ds.close()
    c.vertex_points -= np.float32(0.5)
    s.run("ccs_RefineVertexPoints_Scatter")
    check(O.ALL)
    s.close()
