"""The block Jacobi SVD at the edges of its row chunks (128 rows per chunk of
the workgroup) and column blocks, its relative accuracy on graded matrices,
and where nothing is to be rotated."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

EPS = np.finfo(float).eps


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from parla_amd import ops
    ops.lib()
    return ops


@pytest.mark.parametrize("m,n", [(1, 1), (2, 2), (16, 15), (17, 16), (33, 17), (127, 100), (128, 128), (129, 129),
                                 (257, 90), (385, 40), (400, 385), (641, 33), (1024, 20)])
def test_round_edges(ops, m, n):
    print(f"[gpu-jacobi-rounds] {m} x {n}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, n)) * np.logspace(0, -3, n)
    U, s, Vt = (t.cpu().numpy() for t in ops.svd_jacobi(torch.from_numpy(A).cuda()))
    ref = np.linalg.svd(A, compute_uv=False)
    assert np.all(np.diff(s) <= 0)
    # each sweep rounds every column once per round: 20 sweeps, m-term products
    tol = 50 * EPS * max(m, 16)
    assert np.max(np.abs(s - ref)) <= tol * ref[0]
    assert np.linalg.norm(U.T @ U - np.eye(n)) <= tol * n
    assert np.linalg.norm(Vt @ Vt.T - np.eye(n)) <= tol * n
    assert np.linalg.norm(U * s @ Vt - A) <= tol * np.linalg.norm(A)


def _singular_values_extended(A):
    """One-sided Jacobi in extended precision (64 bits): relative accuracy of order 1e-19 times the condition
    number of A's columns scaled to unit length."""
    W = A.astype(np.longdouble)
    n = W.shape[1]
    tol = 16 * np.finfo(np.longdouble).eps
    for _ in range(40):
        rotated = False
        for p in range(n - 1):
            for q in range(p + 1, n):
                al, be, ga = W[:, p] @ W[:, p], W[:, q] @ W[:, q], W[:, p] @ W[:, q]
                if abs(ga) <= tol * np.sqrt(al * be):
                    continue
                rotated = True
                zeta = (be - al) / (2 * ga)
                t = (1 if zeta >= 0 else -1) / (abs(zeta) + np.sqrt(1 + zeta * zeta))
                c = 1 / np.sqrt(1 + t * t)
                W[:, p], W[:, q] = c * W[:, p] - c * t * W[:, q], c * t * W[:, p] + c * W[:, q]
        if not rotated:
            return np.sort(np.sqrt((W * W).sum(0)))[::-1].astype(np.float64)
    raise AssertionError("no convergence")


@pytest.mark.parametrize("m,n,order", [(57, 48, "permuted"), (57, 48, "descending"), (57, 48, "ascending"),
                                       (24, 16, "permuted")])
def test_graded_columns_keep_relative_accuracy(ops, m, n, order):
    """Gaussian columns scaled from 1 to 1e-14: every pair is rotated, and as
    the columns are well conditioned once scaled to unit length, one-sided
    Jacobi determines every singular value to high relative accuracy (Demmel
    and Veselic 1992)."""
    print(f"[gpu-jacobi-rounds] graded {m} x {n} {order}", flush=True)
    rng = np.random.default_rng(2)
    G = rng.standard_normal((m, n))
    scale = np.logspace(0, -14, n)
    scale = {"permuted": rng.permutation(scale), "descending": scale, "ascending": scale[::-1]}[order]
    A = G * scale
    C = np.abs((A.T @ A) / np.outer(np.linalg.norm(A, axis=0), np.linalg.norm(A, axis=0)) - np.eye(n))
    assert np.median(C) > 1e-2                  # the angles are far above the rotation threshold m eps
    U, s, Vt = (t.cpu().numpy() for t in ops.svd_jacobi(torch.from_numpy(np.ascontiguousarray(A)).cuda()))
    ref = _singular_values_extended(A)
    # one-sided Jacobi: a few rounding errors per round and column, times the scaled condition number
    kappa = np.linalg.cond(G / np.linalg.norm(G, axis=0))
    assert np.max(np.abs(s - ref) / ref) <= n * EPS * kappa
    tol = 50 * EPS * max(m, 16)
    assert np.linalg.norm(U.T @ U - np.eye(n)) <= tol * n
    assert np.linalg.norm(Vt @ Vt.T - np.eye(n)) <= tol * n


@pytest.mark.parametrize("scale", [[1e80, 1e50, 1e20, 1.0], [1e76], [1e-74], [1e-78], [1e-80], [1e70, 1e-70]])
def test_rotations_over_a_wide_range(ops, scale):
    """Column lengths far from 1, alone and side by side: the accumulated
    rotation is one (the squared lengths stay inside FP64, their products'
    squares do not), and so are the singular vectors that do not need lengths
    whose squares underflow."""
    print(f"[gpu-jacobi-rounds] scale {scale}", flush=True)
    m, n = 24, 16
    A = np.random.default_rng(0).standard_normal((m, n)) * np.resize(np.asarray(scale), n)
    U, s, Vt = (t.cpu().numpy() for t in ops.svd_jacobi(torch.from_numpy(A).cuda()))
    tol = 50 * EPS * max(m, 16)
    assert np.linalg.norm(Vt @ Vt.T - np.eye(n)) <= tol * n
    if min(scale) >= 1e-70:
        assert np.linalg.norm(U.T @ U - np.eye(n)) <= tol * n
        ref = np.linalg.svd(A, compute_uv=False)
        assert abs(s[0] - ref[0]) <= tol * ref[0]


@pytest.mark.parametrize("m,n", [(17, 16), (40, 12), (300, 30), (30, 300), (200, 100)])
@pytest.mark.parametrize("kind", ["one column repeated", "ones", "outer", "two of each"])
def test_rank_deficient_matrices_down_to_underflow(ops, m, n, kind):
    """Equal columns leave a QR factor with rows of length 1e-16, 1e-32, ..,
    down to subnormal numbers: the sweeps end, the singular values that are
    not rounding errors are right, and so is the product."""
    print(f"[gpu-jacobi-rounds] {kind} {m} x {n}", flush=True)
    rng = np.random.default_rng(0)
    X = rng.standard_normal((m, n))
    A = {"one column repeated": np.repeat(X[:, :1], n, axis=1), "ones": np.ones((m, n)),
         "outer": np.outer(X[:, 0], X[0]), "two of each": np.repeat(X[:, :(n + 1) // 2], 2, axis=1)[:, :n]}[kind]
    U, s, Vh = (t.cpu().numpy() for t in ops.thin_svd(torch.from_numpy(np.ascontiguousarray(A)).cuda()))
    tol = 50 * EPS * max(m, n, 16)
    assert np.max(np.abs(s - np.linalg.svd(A, compute_uv=False))) <= tol * s[0]
    assert np.linalg.norm((U * s) @ Vh - A) <= tol * np.linalg.norm(A)


def test_orthogonal_columns_are_left_alone(ops):
    n = 40
    A = np.zeros((n + 3, n))
    A[np.arange(n), np.arange(n)] = np.linspace(2.0, 1.0, n)
    U, s, Vt = (t.cpu().numpy() for t in ops.svd_jacobi(torch.from_numpy(A).cuda()))
    np.testing.assert_allclose(s, np.linspace(2.0, 1.0, n), rtol=4 * EPS)
    np.testing.assert_array_equal(np.abs(Vt), np.eye(n))
