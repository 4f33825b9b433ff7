"""The closest-point walk at the numbers of queries where its waves change shape, and with box
distances that only an exact comparison tells apart: bit for bit what each query gives alone and
what the oracle gives."""
import numpy as np
import pytest

import oracle_py as O

pytestmark = pytest.mark.gpu


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("nq", [1, 7, 16, 17, 2047, 2048, 2049, 4095, 4096, 4097, 8192, 8193, 16384, 16385])
def test_number_of_queries(nq):
    from pyhexopt import capi, meshgen as mg
    SV, SF = mg.superellipsoid(3)
    s = capi.Surface(SV, SF)
    rng = np.random.default_rng(1)
    P = rng.uniform(-1.2, 1.2, size=(16385, 3))
    P[::5] = SV[rng.integers(0, SV.shape[0], size=P[::5].shape[0])]        # on vertices: many faces tie
    all_ = s.closest(P)
    part = s.closest(P[:nq])
    assert same(part, [x[:nq] for x in all_])
    FN, VN, FEN = capi.surface_normals(SV, SF)
    S, I, C, N, _ = O.signed_distance_pseudonormal(P[:nq], SV, SF, FN, VN, FEN)
    assert same(part, (S, I, C, N))


@pytest.mark.parametrize("scale", [1.0, 1e-25, 1e12])
def test_near_ties_and_scales(scale):
    """A lattice of coplanar triangles and queries a few ulps off its symmetry planes (box distances
    equal or next to equal), at scales where squared distances leave the float range."""
    from pyhexopt import capi, meshgen as mg
    SV, SF = mg.cube_surface(6)
    SV = SV * scale
    rng = np.random.default_rng(4)
    g = rng.integers(-2, 15, size=(3000, 3)) / 12.0
    P = (g + rng.integers(-2, 3, size=g.shape) * 2.0 ** -52) * scale
    FN, VN, FEN = capi.surface_normals(SV, SF)
    S, I, C, N, _ = O.signed_distance_pseudonormal(P, SV, SF, FN, VN, FEN)
    assert same(capi.Surface(SV, SF).closest(P), (S, I, C, N))


def test_queries_that_are_not_finite():
    from pyhexopt import capi, meshgen as mg
    SV, SF = mg.cube_surface(2)
    P = np.array([[np.nan, 0, 0], [np.inf, 0, 0], [0.5, 0.5, 0.4], [0, -np.inf, np.nan]])
    S, I, C, N = capi.Surface(SV, SF).closest(P)
    assert np.isnan(S[[0, 3]]).all() and (I[[0, 3]] == -1).all() and np.isfinite(S[2]) and I[2] >= 0
