"""The symmetric-Dirichlet local step against its definition, tet by tet: single hexes whose
corner tets all have one known Jacobian U diag(s) V^T, over singular values where the weights
change form or lose digits (undeformed, inside and just outside the band |s - 1| < 1e-8,
ill-conditioned, inverted) and on both reference operators (cube, general)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# singular values (the last one negated: inverted)
SIGMA = [(1, 1, 1), (1 + 5e-9, 1, 1 - 5e-9), (1 + 1.5e-8, 1.1, 0.9), (1 + 3e-8, 1.2, 0.7), (1.3, 1 - 1e-6, 0.8),
         (1.4, 1, 0.6), (1 + 1e-4, 1 + 2e-5, 1 - 3e-5), (2, 1.3, 0.5), (1.7, 1.7, 0.4), (30, 8, 0.05), (12, 1.5, 0.004),
         (1.2, 1.1, -0.7), (3, 0.9, -1e-3)]
EPS = np.finfo(float).eps


def rotation(rng):
    q, r = np.linalg.qr(rng.normal(size=(3, 3)))
    q = q * np.sign(np.diag(r))
    return q if np.linalg.det(q) > 0 else q[:, [1, 0, 2]]


def weight2(s):
    """The reference's squared weight of singular value s, in a form without cancellation."""
    return 1.0 if abs(s - 1) < 1e-8 else (s + 1) * (s * s + 1) / s ** 3


@pytest.mark.parametrize("cube", [True, False])
def test_weights_rhs_and_diagonal(cube):
    from pyhexopt import capi, meshgen as mg
    rng = np.random.default_rng(11)
    nH = len(SIGMA) * 25                       # 325 hexes: several tiles, the last one partly filled
    box = mg.HEX_CORNERS - 0.5
    V = np.tile(box, (nH, 1))
    H = np.arange(8 * nH, dtype=np.int32).reshape(nH, 8)
    A, want, rot, kappa, near = [], [], [], [], []
    for h in range(nH):
        s = np.array(SIGMA[h % len(SIGMA)], dtype=float)
        U, W = rotation(rng), rotation(rng)
        A.append(U @ np.diag(s) @ W.T)
        a = np.abs(s)
        want.append(U @ np.diag([weight2(x) for x in a]) @ U.T)
        # the closest rotation: an inverted tet's smallest direction is flipped back
        rot.append(U @ W.T)
        kappa.append(a.max() / a.min())
        # distance from 1 of the singular value nearest to it outside the band
        near.append(min([abs(x - 1) for x in a if abs(x - 1) >= 1e-8], default=np.inf))
    A, want, rot, kappa, near = (np.array(x) for x in (A, want, rot, kappa, near))
    X = np.einsum("hij,hkj->hki", A, V.reshape(nH, 8, 3)).reshape(-1, 3)
    h = capi.HexOpt(V, H)
    h.reference(cube=cube)
    h.set_positions(capi.CURRENT, X)
    K = h.debug_operator()
    # a unit cube's corner tets have reference factor 1, so K is W^2 (and a general reference
    # operator turns the axes of J's right side only, which W does not see)
    got = K[:, :, [0, 3, 4, 3, 1, 5, 4, 5, 2]].reshape(nH, 8, 3, 3)
    scale = np.abs(want).max(axis=(1, 2))
    err = np.abs(got - want[:, None]).max(axis=(1, 2, 3)) / scale
    # J's entries carry an error of a few eps |J|, which moves 1/s by that times kappa and its cube by
    # three times as much; the reference's form of the weight, (s - s^-3) / (s - 1), rounds its
    # numerator to a few eps and divides it by s - 1
    tol = 60 * EPS * kappa + 4 * EPS / near
    assert (err < tol).all(), (err / tol).max()
    prox = 1e-5
    rhs, invd, _ = h.debug_system(X.T.reshape(-1))
    rhs, diag = rhs.reshape(3, -1).T.reshape(nH, 8, 3), 1.0 / invd.reshape(3, -1).T.reshape(nH, 8, 3)
    Z = want @ rot
    frhs, fdiag = np.zeros((nH, 8, 3)), np.zeros((nH, 8, 3))
    d = np.diagonal(want, axis1=1, axis2=2)
    for t in mg.HEX_TETRA_TABLE:
        for k in t[1:]:
            e = (mg.HEX_CORNERS[k] - mg.HEX_CORNERS[t[0]]).astype(float)   # the edge in the reference
            frhs[:, k] += Z @ e
            frhs[:, t[0]] -= Z @ e
            fdiag[:, k] += d
        fdiag[:, t[0]] += 3 * d
    assert (np.abs(diag - fdiag - prox).max(axis=(1, 2)) < 10 * tol * scale).all()
    # the closest rotation moves by eps kappa as well; X enters with the proximal term
    assert (np.abs(rhs - frhs - prox * X.reshape(nH, 8, 3)).max(axis=(1, 2)) < 20 * tol * scale).all()
