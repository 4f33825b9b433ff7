"""Rows handed in and out (positions, gradients, Hessian-vector products) keep the caller's
numbering: bit for bit on meshes whose vertices the layout renumbers, at sizes around a block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 5, 6])       # 8, 27, 216 and 343 vertices
def test_positions_round_trip(n):
    from pyhexopt import capi, meshgen as mg
    rng = np.random.default_rng(n)
    V, H = mg.grid_hex(n)
    perm = rng.permutation(V.shape[0])               # the caller's numbering follows nothing
    inv = np.argsort(perm)
    h = capi.HexOpt(V[perm], inv[H].astype(np.int32))
    assert np.array_equal(h.get_positions(capi.REST), V[perm])
    X = rng.normal(size=V.shape)
    X[0], X[-1, 1] = [np.inf, -0.0, np.nan], 5e-324
    h.set_positions(capi.CURRENT, X)
    assert np.array_equal(h.get_positions().view(np.int64), X.view(np.int64))
    assert np.array_equal(h.get_positions(capi.REST), V[perm])


@pytest.mark.parametrize("precision", [32, 64])
def test_gradient_and_hessian_rows_follow_the_numbering(precision):
    from pyhexopt import capi, meshgen as mg
    rng = np.random.default_rng(3)
    V, H = mg.grid_hex(6)
    X = V + rng.normal(0, 0.02, size=V.shape)
    v = rng.normal(size=V.shape)
    perm = rng.permutation(V.shape[0])
    inv = np.argsort(perm)
    a, b = capi.HexOpt(V, H), capi.HexOpt(V[perm], inv[H].astype(np.int32))
    for h in (a, b):
        h.reference()
    # the same sums, taken per vertex in the layout's order: equal up to that order
    eps = np.finfo(np.float64 if precision == 64 else np.float32).eps
    for f in (lambda h, p: h.energy_grad(X[p], precision), lambda h, p: h.hvp(X[p], v[p], precision)):
        ga, gb = f(a, np.arange(V.shape[0])), f(b, perm)
        assert np.abs(gb - ga[perm]).max() <= 64 * eps * np.abs(ga).max()
