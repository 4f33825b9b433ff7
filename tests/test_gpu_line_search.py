"""The line search's energies, which are formed with the bound in one launch and read back with it:
those of the accepted step have to be the energies of the positions that the solve returns. Those of
the start are not returned: they decide which step is accepted, so the steps taken have to be the
ones that the energies of the given positions ask for."""
import numpy as np
import pytest

from pyhexopt import capi, meshgen as mg

pytestmark = pytest.mark.gpu

# The kernel evaluates x + s (y - x), the solve stores the same expression: they differ by a
# rounding of each coordinate (1.1e-16 of up to 1.5) on edges of at least 2/7, a strain of 1.2e-15.
# With singular values above 0.2 the energy changes by at most 2 (1 + 125) times that, and a tree
# sum over the elements adds about 1e-14.
RTOL = 1e-12


def _mesh(n, sigma, planes):
    V, H = mg.grid_hex(n)
    inner = ~mg.grid_boundary_mask(n)
    X = mg.jitter(V, inner, sigma * 2.0 / n, seed=n)
    h = capi.HexOpt(V, H)
    ids = np.nonzero(mg.grid_boundary_mask(n))[0].astype(np.int32)
    if planes:
        N = np.random.default_rng(3).normal(size=(ids.size, 3))
        N /= np.linalg.norm(N, axis=1, keepdims=True)
        h.set_constraints(idsT=ids, normalT=N, disT=(N * V[ids]).sum(1) * 1.1, lamT=1.0)
    h.rest_from_current()
    h.reference()
    h.set_positions(capi.CURRENT, X)
    return h, X


def _energy(h):
    E, Eq, Es, _, _ = h.slim_solve(0, weight_opt=1.0)
    return np.array([E, Eq, Es])


# 6 and 7: blocks that are not full; 1: one hex, whose interior is empty. The hex held by planes and
# the two starts with inverted or nearly flat tets reject the step bound (the latter in FP64 only)
@pytest.mark.parametrize("n,sigma,planes,rejects", [
    (1, 0.15, False, ()), (1, 0.15, True, (64, 32)), (6, 0.15, False, ()), (6, 0.15, True, ()), (7, 0.15, False, ()),
    (7, 0.15, True, ()), (6, 0.4, True, (64,)), (7, 0.3, False, (64,))])
@pytest.mark.parametrize("precision", [64, 32])
def test_energies_of_the_accepted_step(n, sigma, planes, rejects, precision):
    h, X = _mesh(n, sigma, planes)
    start = _energy(h)
    assert np.array_equal(h.get_positions(), X)
    if precision == 64:
        E, Eq, Es, log, _ = h.slim_solve(1, weight_opt=1.0)
        assert np.allclose([E, Eq, Es], log[0, :3], rtol=0, atol=0)
    else:
        E, log = h.opt32_solve(1, weight_opt=1.0, residual_every=0)
        assert E == log[0, 0]
    after, Y = _energy(h), h.get_positions()
    bound, step = log[0, 3], log[0, 4]
    # the starts with nearly flat tets: a mean energy of 9,000 over 1,728 tets that comes from a few has
    # singular values down to 2e-4, where the strain above moves it by 1e-11
    rtol = RTOL if sigma == 0.15 else 1e-8
    assert np.allclose(log[0, :3], after, rtol=rtol, atol=rtol * after[1])
    assert after[0] <= start[0] * (1 + rtol)
    assert 0 <= step <= bound <= 1
    if n > 1 or planes:  # (the lone hex without planes starts at its minimum)
        assert step > 0
    if step > 0:  # the bound, or the bound halved some times
        k = np.log2(bound / step)
        assert abs(k - round(k)) < 1e-12
    assert (step < bound) == (precision in rejects)
    if 0 < step < bound:  # the step tried before, twice as long, raised the energy
        h.set_positions(capi.CURRENT, X + 2 * (Y - X))
        assert _energy(h)[0] > start[0]
