"""The packed triangular solves and the LSQR iteration built on them, at the
edges of their 64-row blocks, of one / two block rows per wavefront (512) and
of the packed form (1024)."""
import sys

import numpy as np
import pytest
import scipy.linalg as la

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


@pytest.mark.parametrize("n", [1, 7, 8, 9, 16, 17, 63, 64, 65, 128, 200, 511, 512, 513, 577, 1000, 1024])
def test_packed_solves(ops, n):
    print(f"[gpu-trsv-packed] n={n}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(n)
    R = np.triu(rng.standard_normal((n, n))) + np.diag(3 + np.sqrt(n) + rng.random(n))
    wide = rng.standard_normal((n, n + 3)) * 1e3     # ld > n, junk below the diagonal
    wide[:, :n] = R + np.tril(wide[:, :n], -1)
    Rd = torch.from_numpy(wide).cuda()[:, :n]
    tri = ops.TriSolver(Rd)
    for trans in (False, True):
        b = rng.standard_normal(n)
        x = tri.solve_(torch.from_numpy(b.copy()).cuda(), trans).cpu().numpy()
        Rop = R.T if trans else R
        # backward error of a blocked solve with inverted 8 x 8 diagonal blocks (well conditioned here)
        assert la.norm(Rop @ x - b) <= 10 * n * EPS * la.norm(R) * la.norm(x)


@pytest.mark.parametrize("n", [1, 40, 64, 65, 512, 513, 1024, 1025])
@pytest.mark.parametrize("rows", [2, 9])
@pytest.mark.parametrize("sqrt_delta", [0.0, 0.5])
def test_lsqr_around_the_packed_limits(ops, n, rows, sqrt_delta):
    """rows = 2 / 9 rows per column: few enough pass partials for the tail to
    sum itself at small n, and the reduction kernel.  R comes from a
    perturbed Gram matrix, so a few iterations are needed."""
    print(f"[gpu-trsv-packed] lsqr n={n} rows={rows} delta={sqrt_delta}", flush=True)
    sys.stdout.flush()
    m = rows * n + 3
    rng = np.random.default_rng(n * rows)
    A = rng.standard_normal((m, n)) / np.sqrt(m)
    b = A @ rng.standard_normal(n) + 0.1 * rng.standard_normal(m)
    AL = np.vstack([A, sqrt_delta * np.eye(n)]) if sqrt_delta else A
    bL = np.concatenate([b, np.zeros(n)]) if sqrt_delta else b
    ref = la.lstsq(AL, bL)[0]
    R = la.cholesky(AL.T @ AL + 0.1 * np.diag(rng.random(n)))
    x, xo, _, _, res = ops.lsqr_run(torch.from_numpy(A).cuda(), torch.from_numpy(b).cuda(),
                                    R=torch.from_numpy(np.ascontiguousarray(R)).cuda(), sqrt_delta=sqrt_delta,
                                    atol=1e-14, btol=1e-14, conlim=0.0, iter_lim=200, want_orig=True)
    xo, x = xo.cpu().numpy(), x.cpu().numpy()
    assert la.norm(R @ xo - x) <= 100 * n * EPS * la.norm(R) * la.norm(xo)
    # kappa(A) < 20 and the gradient is reduced to rounding level: an error of order kappa^2 n u
    assert la.norm(xo - ref) <= 400 * 10 * n * EPS * la.norm(ref) + 1e-10 * la.norm(ref), (res.istop, res.itn)
