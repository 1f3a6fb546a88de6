"""The register-resident Cholesky factorisation at the edges of its 16 x 16
tiles, of its instantiations (128, 208) and of the blocked form's steps (128
rows while more than 208 are left), with failing pivots, single and batched."""
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


def _gram(n, rng, spread):
    Y = rng.standard_normal((n + 20, n)) * np.logspace(0, -spread, n)
    return Y.T @ Y


def _check(R, G, n):
    # backward error of a Cholesky factorisation: |R^T R - G| <= c n u |R^T||R|
    B = np.abs(R.T) @ np.abs(R)
    assert np.all(np.abs(R.T @ R - G) <= 4 * (n + 8) * EPS * B)


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 127, 128, 129, 208, 209, 266, 336, 337, 464, 465, 511, 512])
@pytest.mark.parametrize("spread", [0, 4])
def test_potrf_edges(ops, n, spread):
    print(f"[gpu-potrf] n={n} spread={spread}", flush=True)
    sys.stdout.flush()
    rng = np.random.default_rng(n)
    G = _gram(n, rng, spread)
    wide = rng.standard_normal((n, n + 5))       # lda > n; the strictly lower part is neither read nor written
    wide[:, :n] = np.triu(G) + np.tril(wide[:, :n], -1)
    M = torch.from_numpy(wide).cuda()
    info = torch.full((1,), 7, dtype=torch.int32, device="cuda")
    ops.potrf_(M[:, :n], info)
    out = M.cpu().numpy()
    assert int(info.item()) == 0
    _check(np.triu(out[:, :n]), G, n)
    np.testing.assert_array_equal(np.tril(out[:, :n], -1), np.tril(wide[:, :n], -1))
    np.testing.assert_array_equal(out[:, n:], wide[:, n:])


@pytest.mark.parametrize("n,bad", [(1, 1), (16, 9), (17, 17), (100, 48), (266, 266), (266, 128), (266, 129), (289, 3), (512, 256),
                                   (512, 257), (512, 400), (512, 512)])
@pytest.mark.parametrize("value", [-1.0, 0.0, np.nan, np.inf])
def test_potrf_reports_the_failing_pivot(ops, n, bad, value):
    print(f"[gpu-potrf] n={n} bad={bad} value={value}", flush=True)
    sys.stdout.flush()
    G = np.eye(n) * 2.0
    G[bad - 1, bad - 1] = value
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    ops.potrf_(torch.from_numpy(G).cuda(), info)
    assert int(info.item()) == bad


def test_potrf_batched_mixed_sizes(ops):
    rng = np.random.default_rng(5)
    ns = [1, 40, 128, 129, 208, 209, 336, 337, 512, 512, 300, 16]
    fail = {4: 100, 10: 290}
    Gs = []
    for i, n in enumerate(ns):
        G = _gram(n, rng, 2)
        if i in fail:
            G[fail[i] - 1, fail[i] - 1] = -1.0
        Gs.append(G)
    off = np.concatenate([[0], np.cumsum([n * n for n in ns])])
    pool = torch.from_numpy(np.concatenate([np.triu(G).reshape(-1) for G in Gs])).cuda()
    nv = torch.tensor(ns, dtype=torch.int64, device="cuda")
    od = torch.from_numpy(off[:-1].copy()).cuda()
    info = torch.full((len(ns),), 7, dtype=torch.int32, device="cuda")
    ops.check(ops.lib().pamd_potrf_batched_f64(len(ns), ops._p(nv), ops._p(od), ops._p(pool), ops._p(info),
                                               ops.stream(pool.device)), "pamd_potrf_batched_f64")
    inf, host = info.cpu().numpy(), pool.cpu().numpy()
    for i, n in enumerate(ns):
        assert inf[i] == fail.get(i, 0)
        if i not in fail:
            _check(host[off[i]:off[i + 1]].reshape(n, n), Gs[i], n)


@pytest.mark.parametrize("ns", [[0, 1, 16, 128], [129, 128, 5], [208, 130, 0, 208], [209, 3], [336, 337, 128, 129, 210],
                                [512, 1, 465, 400, 209, 208], [512] * 3])
def test_potrf_batched_with_the_largest_size(ops, ns):
    """The form that is given the largest size launches the steps it needs and
    gives the bits of the other one, failing pivots included."""
    print(f"[gpu-potrf] batched ns={ns}", flush=True)
    rng = np.random.default_rng(len(ns))
    Gs = [_gram(n, rng, 2) if n else np.zeros((0, 0)) for n in ns]
    if ns[0] > 200:
        Gs[0][180, 180] = -1.0
    off = np.concatenate([[0], np.cumsum([n * n for n in ns])])
    start = torch.from_numpy(np.concatenate([np.triu(G).reshape(-1) for G in Gs])).cuda()
    nv, od = torch.tensor(ns, dtype=torch.int64, device="cuda"), torch.from_numpy(off[:-1].copy()).cuda()
    L, st, out = ops.lib(), ops.stream(start.device), []
    for nmax in (None, max(ns)):
        pool, info = start.clone(), torch.full((len(ns),), 7, dtype=torch.int32, device="cuda")
        if nmax is None:
            ops.check(L.pamd_potrf_batched_f64(len(ns), ops._p(nv), ops._p(od), ops._p(pool), ops._p(info), st),
                      "pamd_potrf_batched_f64")
        else:
            ops.check(L.pamd_potrf_batched_nmax_f64(len(ns), nmax, ops._p(nv), ops._p(od), ops._p(pool),
                                                    ops._p(info), st), "pamd_potrf_batched_nmax_f64")
        out.append((pool, info))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    for i, n in enumerate(ns):
        bad = 181 if i == 0 and ns[0] > 200 else 0
        assert int(out[0][1][i]) == bad
        if not bad:
            _check(out[0][0][off[i]:off[i + 1]].reshape(n, n).cpu().numpy(), Gs[i], n)
