"""hexopt_octree_copy reads the results from the device: every subset of them, more than once, after
the surface has gone, and after a refinement that failed or grew them."""
import ctypes as C

import numpy as np
import pytest

from pyhexopt import capi, meshgen as mg

pytestmark = pytest.mark.gpu


def _octree(voxels):
    V, F = mg.icosphere(3)
    vs, origin, grid, mt = mg.octree_frame(V, voxels)
    s = capi.Surface(V, F)
    return s, capi.Octree(s, grid, origin, vs, mt, 1)


@pytest.mark.parametrize("voxels", [2, 17, 64])
def test_copy_subsets_after_the_surface(voxels):
    s, o = _octree(voxels)
    r = o.result()
    del s
    again = o.result()
    names = ("leaves", "nodes", "V", "H")
    for k in names:
        assert np.array_equal(r[k], again[k])
        part = np.zeros_like(r[k])
        args = [part.ctypes.data if j == k else None for j in names]
        assert capi.lib().hexopt_octree_copy(C.c_void_p(o.h), *args) == 0
        assert np.array_equal(part, r[k])
    assert capi.lib().hexopt_octree_copy(C.c_void_p(o.h), None, None, None, None) == 0
    o.close()


def test_copy_around_refine():
    s, o = _octree(64)
    r = o.result()
    with pytest.raises(RuntimeError):
        o.refine(s, 1, [[1, 1, 1, 3]])
    kept = o.result()
    assert all(np.array_equal(r[k], kept[k]) for k in ("leaves", "nodes", "V", "H"))
    big = r["leaves"][r["leaves"][:, 3] > 1][:50]
    o.refine(s, 0, big)
    grown = o.result()
    assert grown["H"].max() < len(grown["V"]) and len(grown["leaves"]) >= len(r["leaves"])
    p = grown["nodes"][grown["H"][:, 0]]
    assert np.array_equal(p.min(0), r["nodes"][r["H"][:, 0]].min(0))
    o.close()
