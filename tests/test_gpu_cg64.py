"""The FP64 CG of slim_solve against the same 20 steps in numpy on the operator of
hexopt_debug_system: one partly filled tile, several tiles, feature lines, a vertex without hexes,
both reference operators."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,lines,loose,cube", [(2, False, False, True), (6, True, False, True), (7, True, True, True),
                                                (9, False, False, True), (7, True, True, False)])
def test_direction_is_twenty_cg_steps(n, lines, loose, cube):
    from pyhexopt import capi, meshgen as mg
    rng = np.random.default_rng(n)
    V, H = mg.grid_hex(n)
    V0 = V + rng.normal(0, 0.05 * 2 / n, size=V.shape)
    bnd = np.nonzero(mg.grid_boundary_mask(n))[0].astype(np.int32)
    if loose:                                        # a vertex that belongs to no hex, held by its plane
        V0 = np.concatenate([V0, [[2.0, 0.1, 0.3]]])
        bnd = np.concatenate([bnd, [V.shape[0]]]).astype(np.int32)
    nL = 9 if lines else 0
    idsL, idsT = bnd[:nL], bnd[nL:]
    N, T = rng.normal(size=(idsT.size, 3)), rng.normal(size=(nL, 3))
    N /= np.linalg.norm(N, axis=1)[:, None]
    T /= np.linalg.norm(T, axis=1)[:, None]
    h = capi.HexOpt(V0, H)
    h.reference(cube=cube)
    h.set_constraints(idsT=idsT, normalT=N, disT=(N * V0[idsT]).sum(1) + rng.normal(0, 0.02, size=idsT.size), lamT=3.0,
                      idsL=idsL, axaL=T, originL=V0[idsL] + rng.normal(0, 0.02, size=(nL, 3)), lamL=2.0)
    nV = V0.shape[0]
    x = np.concatenate([V0.T.ravel(), np.zeros(nL)])
    rhs, inv, Lx = h.debug_system(x)
    r = rhs - Lx
    p = inv * r
    new, its = r @ p, 0
    for _ in range(20):
        Lp = h.debug_system(p)[2]
        alpha = new / (p @ Lp)
        x, r = x + alpha * p, r - alpha * Lp
        if r @ r < 1e-16 * (rhs @ rhs):
            break
        z = inv * r
        old, new = new, r @ z
        p, its = z + new / old * p, its + 1
    E, Eq, Es, log, aL = h.slim_solve(1)
    step = log[0, 4]
    assert step > 0 and int(log[0, 5]) == its
    d = (h.get_positions() - V0) / step
    want = (x[:3 * nV].reshape(3, -1).T - V0)
    # 20 steps amplify the rounding of the sums by some powers of ten; the direction's own size is
    # the scale (the positions carry eps |V| / step)
    tol = 1e-9 * np.abs(want).max()
    held = V.shape[0]
    assert np.abs(d - want)[:held].max() < tol
    if loose:
        # the loose vertex is a block of its own. Across its plane diag^-1 L has the eigenvalue 3, the
        # largest there is: with steps of about 1 each CG step doubles what rounding left there
        # (2^20 eps |x| after 20), and along the plane only the proximal term (1e-5) holds it, so
        # the rounding of lamT n (n.x) moves it by eps lamT |x| / 1e-5
        eps = np.finfo(float).eps
        assert np.abs((d - want)[held]).max() < 4 * eps * 2.0 * (2 ** 20 + 3.0 / 1e-5)
    assert lines is False or np.abs(aL - x[3 * nV:]).max() < tol + 1e-9 * np.abs(x[3 * nV:]).max()
    assert log[0, 6] == pytest.approx(np.sqrt(r @ r / (rhs @ rhs)), rel=1e-5)
