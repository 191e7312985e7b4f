"""The block eigensolver on both sides of the order from which its matrix
leaves LDS (131/132), at the edges of the 64-entry pieces its waves hold, and
on spectra with repeated eigenvalues, against its own defining equations and
LAPACK.

Tolerance: reduction, QL and back-transformation are products of orthogonal
transformations and triangular solves with a well-conditioned U, so residual,
orthogonality and eigenvalues are within a small multiple of n eps of the
largest eigenvalue (or of 1): 4 (n + 4) eps.
"""
import numpy as np
import pytest
import scipy.linalg

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def problem(n, seed, repeat=0):
    rng = np.random.default_rng(seed)
    v, _ = np.linalg.qr(rng.normal(size=(n, n)))
    e = 100.0 + np.cumsum(rng.uniform(0.1, 4.0, n))
    e[n // 3:n // 3 + repeat] = e[n // 3]
    A = (v * e) @ v.T
    s = rng.normal(size=(n, n)) * 0.1 / np.sqrt(n)
    return 0.5 * (A + A.T), np.eye(n) + 0.5 * (s + s.T)


@pytest.mark.parametrize("n,repeat", [(1, 0), (2, 0), (3, 0), (64, 10),
                                      (131, 0), (132, 0), (133, 40), (192, 0),
                                      (193, 0), (255, 60), (256, 0)])
def test_orders(hip, n, repeat):
    from mlcp_amd import intertwine as tw
    print("[case] gep", n, repeat, flush=True)
    A, B = problem(n, n, repeat)
    w, X = tw.gpu_gep(A, B)
    tol = 4 * (n + 4) * EPS
    scale = np.abs(w).max()
    assert np.max(np.abs(A @ X - B @ X * w)) <= tol * scale
    assert np.max(np.abs(X.T @ B @ X - np.eye(n))) <= tol
    ref = scipy.linalg.eigh(A, B, eigvals_only=True)
    assert np.max(np.abs(w - ref)) <= tol * scale
    assert np.all(np.diff(w) >= 0)
    big = np.argmax(np.abs(X), axis=0)
    assert np.all(X[big, np.arange(n)] > 0)


@pytest.mark.parametrize("n", [131, 200])
def test_refusals(hip, n):
    from mlcp_amd import intertwine as tw
    A, B = problem(n, 3)
    B[n // 2, n // 2] = -1.0
    with pytest.raises(RuntimeError, match="positive definite"):
        tw.gpu_gep(A, B)
    A, B = problem(n, 4)
    A[n - 1, n - 1] = np.nan
    with pytest.raises(RuntimeError, match="non-finite"):
        tw.gpu_gep(A, B)
