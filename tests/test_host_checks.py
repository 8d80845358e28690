"""Library internals that run on the host, compiled for the CPU alone."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from halfedgecatmullclark_amd import build as B
from halfedgecatmullclark_amd import cage as C
from halfedgecatmullclark_amd.abi import MeshView
from oracle import oracle as O
from tests.helpers import permuted, tip_cages, welded_tori
from tests.test_gpu_rare import bipyramid, cone, prism


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host_checks") / "host_checks.so")
    src = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_checks.hip")
    subprocess.run([B.hipcc(), "--offload-host-only", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wl,-Bsymbolic",
                    "-x", "hip", src, "-o", so],
                   check=True, capture_output=True)
    return ctypes.CDLL(so)


def crossed():
    """a torus with the twins of two edges exchanged"""
    c = C.torus(4, 3).copy()
    e = np.flatnonzero(c.halfedges[:, 0] > np.arange(c.H))[:2]
    t = c.halfedges[e, 0].copy()
    c.halfedges[e, 0] = t[::-1]
    return c


# rings 1, simple 2, table 4
@pytest.mark.parametrize("name,cage,want", [
    ("torus", C.torus(4, 3), 7), ("irregular", C.irregular(1, seed=3), 7), ("prism64", prism(64), 7),
    ("cone63", cone(63), 7), ("prism65", prism(65), 3), ("bipyramid65", bipyramid(65), 3), ("cone65", cone(65), 3),
    ("welded", welded_tori(3, 3), 1), ("crossed", crossed(), 1)], ids=lambda x: x if isinstance(x, str) else "")
def test_which_cages_take_the_table_and_the_tiles(checks, name, cage, want):
    m = MeshView(cage.contiguous())
    assert checks.check_rare_table(m.pointer) == want


@pytest.mark.parametrize("i", [0, 1, 2 ** 30 - 1, 1431655765, 1431655766, 2 ** 31 - 1])
def test_record_offsets(checks, i):
    checks.check_at3.restype = ctypes.c_uint64
    for b in (12, 24):
        assert checks.check_at3(i, b, 1) == b * i
        if i < 2 ** 30:
            assert checks.check_at3(i, b, 0) == b * i


def test_lists_without_memory(checks):
    """the threads that build a batch's lists end whichever allocation fails"""
    checks.check_lists.argtypes = [ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64]
    m = MeshView(C.torus(64, 32).contiguous())
    p = ctypes.cast(m.pointer, ctypes.c_void_p)
    assert checks.check_lists(p, 16, -1) == 1
    got = [checks.check_lists(p, 16, k) for k in range(60)]
    assert set(got) <= {0, 1} and 0 in got


@pytest.mark.parametrize("name,cage", [("irregular", C.irregular(5)), ("torus", C.torus(128, 66))],
                         ids=lambda x: x if isinstance(x, str) else "")
def test_lists_on_two_threads(checks, name, cage):
    assert cage.H >= 1 << 15
    assert checks.check_threads(MeshView(cage.contiguous()).pointer)


OWNERS = [("torus", C.torus(5, 3), 0), ("irregular", C.irregular(1, seed=3), 0), ("cone", cone(5), 0),
          ("welded", welded_tori(3, 3), 1), ("permuted_torus", permuted(C.torus(4, 3), 1), 1),
          ("permuted_cone", permuted(cone(7), 2), 1)] + [(n, c, 1) for n, c in tip_cages()]


@pytest.mark.parametrize("name,cage,by_pair", OWNERS, ids=[o[0] for o in OWNERS])
def test_edge_owners(checks, name, cage, by_pair):
    """every edge of every level has one owner, the larger halfedge of its
    pair; the reference's representative where it is that halfedge on every
    level (by_pair 0)"""
    m = MeshView(cage.contiguous())
    out = O.refine(cage, 4, O.HALFEDGES)
    for d in range(1, 5):
        lv = O.level(out, "halfedges", d)
        got = np.full(out["counts"]["E"][d], -1, np.int32)
        assert checks.check_edge_owners(m.pointer, d, ctypes.c_void_p(got.ctypes.data)) == by_pair
        larger = np.flatnonzero(np.arange(len(lv)) > lv["twinID"])
        want = np.full_like(got, -1)
        want[lv["edgeID"][larger]] = larger
        assert np.array_equal(got, want), (d, np.flatnonzero(got != want)[:5])
        if not by_pair:
            assert all(O.edge_to_halfedge(cage, e, d) == got[e] for e in range(0, len(got), 7))
