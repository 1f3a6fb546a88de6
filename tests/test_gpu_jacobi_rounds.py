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


def test_graded_columns_keep_relative_accuracy(ops):
    """Columns scaled from 1 to 1e-14: sigma = D-scaled, well conditioned
    after scaling, so every singular value has relative accuracy."""
    n = 48
    rng = np.random.default_rng(2)
    Q = np.linalg.qr(rng.standard_normal((n + 9, n)))[0]
    # orthogonal columns times a diagonal, mixed by a unit upper triangle close to I
    scale = np.logspace(0, -14, n)
    A = Q * scale
    perm = rng.permutation(n)
    s = ops.svd_jacobi(torch.from_numpy(np.ascontiguousarray(A[:, perm])).cuda())[1].cpu().numpy()
    assert np.max(np.abs(s - scale) / scale) <= 200 * EPS * n


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


def test_orthogonal_columns_are_left_alone(ops):
    n = 40
    A = np.zeros((n + 3, n))
    A[np.arange(n), np.arange(n)] = np.linspace(2.0, 1.0, n)
    U, s, Vt = (t.cpu().numpy() for t in ops.svd_jacobi(torch.from_numpy(A).cuda()))
    np.testing.assert_allclose(s, np.linspace(2.0, 1.0, n), rtol=4 * EPS)
    np.testing.assert_array_equal(np.abs(Vt), np.eye(n))
