"""The matrix-vector passes at the edges of their unrolled loops and launch
rules, and on a matrix past the size from which it is streamed (256 MB):
GEMV both ways, the 2-norm, the LSQR pass, the normal pass, the residual."""
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


def _randn(*shape, seed=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(*shape, dtype=torch.float64, device="cuda", generator=g)


@pytest.mark.parametrize("m,n", [(1, 1), (3, 511), (5, 512), (5, 513), (2048, 2047), (2048, 2048), (2049, 2048),
                                 (7, 20001), (31, 65), (32, 64), (33, 63), (5000, 200), (70000, 512), (35, 65472), (35, 65473)])
def test_gemv(ops, m, n):
    print(f"[gpu-passes] gemv {m} x {n}", flush=True)
    sys.stdout.flush()
    A, x, y = _randn(m, n), _randn(n, seed=1), _randn(m, seed=2)
    scale = float(A.norm()) / np.sqrt(m * n) if m * n > 1 else 1.0
    ref = A @ x
    assert float((ops.gemv(A, x) - ref).norm()) <= 8 * EPS * n * scale * float(x.norm()) * np.sqrt(m)
    out = ops.gemv(A, x, y=y.clone(), alpha=2.0, beta=-1.0)
    assert float((out - (2.0 * ref - y)).norm()) <= 8 * EPS * (n + 1) * (scale * float(x.norm()) * np.sqrt(m)
                                                                         + float(y.norm()))
    assert float((ops.gemv(A, y, trans=True) - A.t() @ y).norm()) <= 8 * EPS * m * scale * float(y.norm()) * np.sqrt(n)


@pytest.mark.parametrize("n", [1, 1024, 8191, 8192, 8193, 32768, 32769, 100000, 100001, 36_000_000])
def test_nrm2(ops, n):
    print(f"[gpu-passes] nrm2 {n}", flush=True)
    sys.stdout.flush()
    x = _randn(n)
    ref = float(x.norm())
    assert abs(float(ops.nrm2(x).item()) - ref) <= 64 * EPS * ref


@pytest.mark.parametrize("m,n", [(1, 1), (4, 3), (63, 20), (64, 20), (65, 65), (16384, 40), (16400, 300), (20001, 513),
                                 (33000, 1024), (70001, 512)])
def test_lsqr_normal_and_residual_passes(ops, m, n):
    """One LSQR run from x = 0 with a single iteration is two passes over A;
    the normal pass and the compensated residual are one each."""
    print(f"[gpu-passes] passes {m} x {n}", flush=True)
    sys.stdout.flush()
    A, b = _randn(m, n), _randn(m, seed=1)
    x, _, _, res = ops.lsqr_run(A, b, atol=0.0, btol=0.0, conlim=0.0, iter_lim=1)
    # x_1 = (v . A^T b) / ||A v||^2 v with v = A^T b / ||A^T b||
    g = A.t() @ b
    v = g / g.norm()
    ref = (g @ v) / (A @ v).square().sum() * v
    # the products with a Gaussian A lose at most a factor of its condition number, bounded by its size here
    assert float((x - ref).norm()) <= 64 * EPS * (m + n) * float(ref.norm())
    p = _randn(n, seed=3)
    q = ops.NormalOp(A)(p)
    assert float((q - A.t() @ (A @ p)).norm()) <= 16 * EPS * np.sqrt(m * n) * float(A.norm()) ** 2 * float(p.norm())
    B = A.to(torch.float32)
    q = ops.NormalOp(B)(p)
    ref = B.double().t() @ (B.double() @ p)
    assert float((q - ref).norm()) <= 16 * EPS * np.sqrt(m * n) * float(A.norm()) ** 2 * float(p.norm())
    gr, rss, r = ops.Residual(A)(p, b, want_r=True)
    rr = b - A @ p
    tol = 16 * EPS * np.sqrt(n) * float(A.norm()) * float(p.norm()) + 16 * EPS * float(b.norm())
    assert float((r - rr).norm()) <= tol
    assert float((gr - A.t() @ rr).norm()) <= tol * float(A.norm()) * 4
    assert abs(float(rss.item()) - float(rr.square().sum())) <= 4 * tol * float(rr.norm()) + 64 * EPS * float(rss.item())


@pytest.mark.parametrize("m,n", [(4096, 513), (4097, 513), (16384, 1024), (32640, 700), (32641, 700), (65537, 600)])
@pytest.mark.parametrize("sqrt_delta", [0.0, 0.3])
def test_lsqr_pass_shapes_without_r(ops, m, n, sqrt_delta):
    """The first iteration without R where the rule for 513..1024 columns
    changes its workgroups, with and without lifted rows."""
    print(f"[gpu-passes] lsqr shape {m} x {n} delta={sqrt_delta}", flush=True)
    A, b = _randn(m, n), _randn(m, seed=1)
    x, _, _, res = ops.lsqr_run(A, b, sqrt_delta=sqrt_delta, atol=0.0, btol=0.0, conlim=0.0, iter_lim=1)
    g = A.t() @ b
    v = g / g.norm()
    ref = (g @ v) / ((A @ v).square().sum() + sqrt_delta ** 2) * v
    assert float((x - ref).norm()) <= 64 * EPS * (m + n) * float(ref.norm())
