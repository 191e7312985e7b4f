"""Vector updates large enough that the right-hand sides read the modes outside
their group through one product array (from six modes and half a GB of cross
Grams on), and the edges of the refresh's column tiles.

All states of the block share their factors and differ in their coefficients,
so every target sum_l U(l, t) Q_l is again a vector of those factors, with the
coefficients C U: the update has to return it.

Tolerance: the fit is exact but for the ALS penalty, 1e-10 of the largest
coefficient on the diagonal of a Gram matrix of nearly orthogonal products
(eigenvalues of order one): relative error below 1e-8 with a factor of a
hundred to spare.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(D, n, B, R, seed):
    from tests.helpers import random_system
    from mlcp_amd.hoplist import CPBlock
    from mlcp_amd.intertwine import Session
    rng = np.random.default_rng(seed)
    fac = rng.normal(size=(R, D, n))
    fac /= np.linalg.norm(fac, axis=2, keepdims=True)
    C = np.exp(rng.uniform(-1.0, 1.0, (R, B)))
    Q = CPBlock(np.full(D, n), np.full(B, R), C.T.ravel().copy(),
                np.tile(fac.reshape(R, D * n), (B, 1)), np.zeros(B))
    H = random_system(seed, [n] * D, ncoup=2)
    U = np.eye(B) + rng.normal(size=(B, B)) * 0.1 / np.sqrt(B)
    with Session(Q, H) as s:
        s.update(U, 2)
        out = s.download()
    G = np.ones((R, R))
    for d in range(D):
        G *= fac[:, d] @ fac[:, d].T
    want = C @ U
    got = out.base.reshape(B, R, D, n)
    for t in range(B):
        # |got - want|^2 over |want|^2, both normalised
        M = np.ones((R, R))
        S = np.ones((R, R))
        for d in range(D):
            M *= got[t, :, d] @ fac[:, d].T
            S *= got[t, :, d] @ got[t, :, d].T
        c = out.coef[t * R:(t + 1) * R]
        ww = want[:, t] @ G @ want[:, t]
        cc = c @ S @ c
        cw = (c @ M @ want[:, t]) / np.sqrt(ww)
        assert abs(cc - 1.0) <= 1e-8
        # 1 - cos^2 of the angle, at rounding level of the products
        assert abs(abs(cw) - 1.0) <= 1e-8


@pytest.mark.parametrize("D,n,B,R", [
    (6, 17, 170, 20),    # 555 MB of cross Grams: groups of three
    (7, 16, 150, 21),    # the last group is one mode
    (12, 9, 130, 18),    # groups of four
])
def test_grouped_products(hip, D, n, B, R):
    print("[case] update groups", D, n, B, R, flush=True)
    assert 8.0 * D * B * R * (B * R) >= 512e6
    check(D, n, B, R, 7 * D + n)


@pytest.mark.parametrize("D,n,B,R", [
    (2, 1, 2, 1), (2, 65, 3, 21), (3, 64, 5, 16), (3, 128, 4, 33),
    (2, 100, 2, 64),
])
def test_column_tiles(hip, D, n, B, R):
    print("[case] update tiles", D, n, B, R, flush=True)
    check(D, n, B, R, n + R)


@pytest.mark.parametrize("n,R,old", [(1, 1, 1), (10, 8, 64), (17, 16, 65),
                                     (33, 33, 128), (33, 33, 129),
                                     (128, 64, 100)])
def test_one_launch_fit(hip, n, R, old):
    """Fits on both sides of two chunks of 64 old columns (one launch or one a
    step): a vector of ``old`` columns that are R products, repeated with other
    coefficients, has to come back as those products."""
    from mlcp_amd.intertwine import gpu_als
    print("[case] fit", n, R, old, flush=True)
    D = 3
    rng = np.random.default_rng(n + old)
    fac = rng.normal(size=(R, D, n))
    fac /= np.linalg.norm(fac, axis=2, keepdims=True)
    which = np.arange(old) % R
    gc = np.exp(rng.uniform(-1.0, 1.0, old))
    want = np.zeros(R)
    np.add.at(want, which, gc)
    F0 = fac.reshape(R, D * n)
    fc, fb = gpu_als(np.ones(R), F0.copy(), gc, F0[which].copy(),
                     np.full(D, n, dtype=np.int32), 2)
    got = np.asarray(fb).reshape(R, D, n)
    S, M, G = np.ones((R, R)), np.ones((R, R)), np.ones((R, R))
    for d in range(D):
        S *= got[:, d] @ got[:, d].T
        M *= got[:, d] @ fac[:, d].T
        G *= fac[:, d] @ fac[:, d].T
    cw = (fc @ M @ want) / np.sqrt((fc @ S @ fc) * (want @ G @ want))
    assert abs(abs(cw) - 1.0) <= 1e-8
