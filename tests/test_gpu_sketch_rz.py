"""R and z = Q^T S b of a sketch by CholeskyQR (pamd_sketch_rz_f64) and the
rule that chooses it: its plain and shifted forms against LAPACK's Householder
QR, columns of very different scales, and a rank-deficient sketch, which ends
at Householder."""
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


def _sketch(d, n, cond, seed):
    rng = np.random.default_rng(seed)
    V = la.qr(rng.standard_normal((n, n)))[0]
    A = (rng.standard_normal((d, n)) / np.sqrt(d) * np.logspace(0, -np.log10(cond), n)) @ V.T
    return np.hstack([A, rng.standard_normal((d, 1))])


def _reference(M, n):
    Q, R = la.qr(M[:, :n], mode="economic")
    s = np.sign(np.diag(R))
    return s[:, None] * R, s * (Q.T @ M[:, n])


@pytest.mark.parametrize("d,n", [(64, 64), (400, 100), (333, 129), (1500, 300), (1100, 513), (1030, 1024)])
@pytest.mark.parametrize("cond,shifted", [(1e3, False), (1e3, True), (1e10, True)])
def test_forms_match_householder(ops, d, n, cond, shifted):
    print(f"[gpu-sketch-rz] d={d} n={n} cond={cond:g} shifted={shifted}", flush=True)
    sys.stdout.flush()
    if d < 2 * n:
        cond = min(cond, 1e8)  # a square Gaussian adds about n to the condition number
    M = _sketch(d, n, cond, d + n)
    kappa = np.linalg.cond(M[:, :n])
    if not shifted and kappa > 1e6:
        pytest.skip("the plain form is for better conditioned sketches")
    rz = ops.sketch_rz_cholqr2(torch.from_numpy(M).cuda(), n, shifted)
    assert rz is not None
    R, z = (t.cpu().numpy() for t in rz)
    Rl, zl = _reference(M, n)
    assert np.all(np.diag(R) > 0) and np.all(np.tril(R, -1) == 0)
    tol = 100 * EPS * kappa * np.sqrt(n)  # two backward stable factorisations
    assert la.norm(R - Rl) <= min(tol, 1e-6) * la.norm(Rl)
    assert la.norm(z - zl) <= tol * la.norm(M[:, n])


@pytest.mark.parametrize("cond", [5e6, 1e7, 1.5e7])
@pytest.mark.parametrize("seed", [1, 2])
def test_solution_between_the_second_rounds(ops, cond, seed):
    """One small singular value, so that ||Q1^T Q1 - I|| is 1e-3 to 1e-2: x =
    R^{-1} z of a consistent system has a backward stable solver's error, a few
    u kappa (the two fixed-point steps alone are off by ||E||^3)."""
    d, n = 800, 200
    print(f"[gpu-sketch-rz] second round cond={cond:g} seed={seed}", flush=True)
    rng = np.random.default_rng(seed)
    V = la.qr(rng.standard_normal((n, n)))[0]
    SA = (rng.standard_normal((d, n)) / np.sqrt(d) * np.r_[np.ones(n - 1), 1.0 / cond]) @ V.T
    x = rng.standard_normal(n)
    M = np.hstack([SA, (SA @ x)[:, None]])
    rz = ops.sketch_rz_cholqr2(torch.from_numpy(M).cuda(), n)
    assert rz is not None
    R, z = (t.cpu().numpy() for t in rz)
    err = la.norm(la.solve_triangular(R, z) - x) / la.norm(x)
    assert err <= 4 * EPS * np.linalg.cond(SA), err


@pytest.mark.parametrize("shifted", [0, 1])
@pytest.mark.parametrize("d,n", [(120, 64), (700, 209), (1100, 513)])
def test_second_round_reuses_the_first(ops, d, n, shifted):
    """newton = 2 gives newton = 0's bits from the workspace that newton = 1
    left, without reading the sketch again."""
    print(f"[gpu-sketch-rz] second round only d={d} n={n} shifted={shifted}", flush=True)
    M = torch.from_numpy(_sketch(d, n, 1e3, 5)).cuda()
    dev = M.device
    L, st = ops.lib(), ops.stream(dev)

    def run(A, newton, ws):
        R, z, stats = (torch.full(s, float("nan"), dtype=torch.float64, device=dev) for s in ((n, n), (n,), (4,)))
        ops.check(L.pamd_sketch_rz_f64(d, n, ops._p(A), n + 1, shifted, newton, ops._p(R), n, ops._p(z),
                                       ops._p(stats), ops._p(ws), st), "pamd_sketch_rz_f64")
        return R, z, stats

    size = ops._query(L.pamd_sketch_rz_workspace, d, n)
    want = run(M, 0, ops.workspace(size, dev))
    ws = ops.workspace(size, dev)
    run(M, 1, ws)
    got = run(torch.full_like(M, float("nan")), 2, ws)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_graded_columns_stay_on_the_plain_form(ops):
    """Cholesky is invariant under column scaling, so scales from 1e-9 to 1e9
    do not matter (R1's diagonal spread is 1e18)."""
    n, d = 120, 500
    M = _sketch(d, n, 10.0, 3)
    M[:, :n] *= np.logspace(-9, 9, n)[np.random.default_rng(1).permutation(n)]
    rz = ops.sketch_rz_cholqr2(torch.from_numpy(M).cuda(), n)
    assert rz is not None
    R, z = (t.cpu().numpy() for t in rz)
    Rl, zl = _reference(M, n)
    scale = la.norm(M[:, :n], axis=0)
    assert np.max(la.norm(R - Rl, axis=0) / scale) <= 1e-12
    assert la.norm(z - zl) <= 1e-12 * la.norm(M[:, n])


@pytest.mark.parametrize("d,n", [(400, 100), (1100, 513)])
def test_nothing_follows_a_failed_pivot(ops, d, n):
    """kappa 1e12 is beyond the Gram matrix: its factorisation fails, which the
    figures report, and the products after it are left out (R is not written)."""
    print(f"[gpu-sketch-rz] failed pivot d={d} n={n}", flush=True)
    M = torch.from_numpy(_sketch(d, n, 1e12, 6)).cuda()
    R = torch.full((n, n), 7.0, dtype=torch.float64, device="cuda")
    z, stats = torch.empty_like(R[0]), torch.empty(4, dtype=torch.float64, device="cuda")
    ws = ops.workspace(ops._query(ops.lib().pamd_sketch_rz_workspace, d, n), M.device)
    ops.check(ops.lib().pamd_sketch_rz_f64(d, n, ops._p(M), n + 1, 0, 1, ops._p(R), n, ops._p(z), ops._p(stats),
                                           ops._p(ws), ops.stream(M.device)), "pamd_sketch_rz_f64")
    assert 1 <= float(stats[3]) <= n
    assert bool((R == 7.0).all())


def test_rank_deficient_sketch_ends_at_householder(ops):
    n, d = 100, 400
    M = _sketch(d, n, 10.0, 4)
    M[:, 50] = M[:, 20] + M[:, 30]
    Md = torch.from_numpy(M).cuda()
    assert ops.sketch_rz_cholqr2(Md, n) is None and ops.sketch_rz_cholqr2(Md, n, True) is None
    np.testing.assert_array_equal(Md.cpu().numpy(), M)
    R, z = (t.cpu().numpy() for t in ops.sketch_rz_(Md, n))
    f = ops.qr_r_(torch.from_numpy(M).cuda(), n)
    np.testing.assert_array_equal(R, f.R().cpu().numpy())
    np.testing.assert_array_equal(z, f.M[:n, n].cpu().numpy())
