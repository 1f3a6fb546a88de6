"""The batched row-block passes, their reduction and the preconditioner products
at the edges of the column groups (64), row groups and row blocks (64), in the
problem's own length class and in the widest one."""
import numpy as np
import pytest
import torch

import oracle as orc

pytestmark = pytest.mark.gpu
U = 2.0 ** -53

# (m, n): one group less, exactly, and one more; last row blocks of 1, 63 and 64 rows; many blocks per problem
SHAPES = [(1, 1), (8, 1), (64, 63), (65, 64), (129, 65), (191, 127), (256, 128), (257, 129), (386, 192), (449, 193),
          (640, 256), (641, 257), (705, 320), (769, 321), (9001, 384), (897, 385), (900, 448), (961, 449), (1100, 511),
          (1537, 512), (20011, 33)]


@pytest.fixture(scope="module")
def batch():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from parla_amd import ops
    import parla_amd.drivers.batched_ls as bl
    ops.lib()
    rng = np.random.default_rng(11)
    As = [rng.standard_normal(s).astype(np.float32) for s in SHAPES]
    bs = [rng.standard_normal(s[0]) for s in SHAPES]
    B = bl.Batch(As, bs, torch.device("cuda"))
    B.t.copy_(torch.from_numpy(rng.standard_normal(B.t.numel())))
    B.x.copy_(torch.from_numpy(rng.standard_normal(B.x.numel())))
    return ops, As, bs, B


def _run(ops, B, kind, wide):
    """One pass over all problems, each in its own class or all in class 8, and its reduction."""
    L, st = ops.lib(), ops.stream(B.dev)
    lists = list(B.blocks.items())
    if wide:
        lists = [(8, torch.cat([b for _, b in lists]).contiguous())]
    B.part.zero_()
    for c, blks in lists:
        if kind == "normal":
            ops.check(L.pamd_bt_normal(c, ops._p(B.desc), ops._p(blks), blks.shape[0], 4, 2, ops._p(B.A), ops._p(B.t),
                                       ops._p(B.state), ops._p(B.part), st), "pamd_bt_normal")
        else:
            ops.check(L.pamd_bt_residual(c, ops._p(B.desc), ops._p(blks), blks.shape[0], 4, 2, ops._p(B.A),
                                         ops._p(B.b), ops._p(B.x), ops._p(B.state), ops._p(B.part), st),
                      "pamd_bt_residual")
    out = torch.full_like(B.g, float("nan"))
    comp = 1 if kind == "residual" else 0
    ops.check(L.pamd_bt_reduce(B.P, ops._p(B.desc), ops._p(B.part), comp, ops._p(out),
                               ops._p(B.rss) if comp else None, st), "pamd_bt_reduce")
    return out


@pytest.mark.parametrize("wide", [False, True], ids=["own class", "class 8"])
def test_normal_pass_edges(batch, wide):
    ops, As, _, B = batch
    print("[bt-passes] normal", wide, flush=True)
    out = _run(ops, B, "normal", wide)
    for i, A in enumerate(As):
        Ad, t = A.astype(np.float64), B.vec(B.t, i).cpu().numpy()
        m, n = A.shape
        # two dot products of lengths n and m, componentwise
        bound = (m + n + 16) * U * (np.abs(Ad).T @ (np.abs(Ad) @ np.abs(t)))
        assert (np.abs(B.vec(out, i).cpu().numpy() - Ad.T @ (Ad @ t)) <= 2 * bound).all(), A.shape


@pytest.mark.parametrize("wide", [False, True], ids=["own class", "class 8"])
def test_residual_pass_edges(batch, wide):
    ops, As, bs, B = batch
    print("[bt-passes] residual", wide, flush=True)
    out = _run(ops, B, "residual", wide)
    rss = B.rss.cpu().numpy()
    for i, (A, b) in enumerate(zip(As, bs)):
        Ad, x = A.astype(np.float64), B.vec(B.x, i).cpu().numpy()
        m, n = A.shape
        _, g, s = orc.residual_exact(Ad, x, b)
        # r correct to u |r| plus second-order terms, g summed in twice the precision: u |A|^T |r| and u |g|
        r = np.abs(b - Ad @ x)
        bound = 2 * U * (np.abs(Ad).T @ r) + 2 * U * np.abs(g) + (m + n) ** 2 * U ** 2 * (
            np.abs(Ad).T @ (np.abs(Ad) @ np.abs(x) + np.abs(b)))
        assert (np.abs(B.vec(out, i).cpu().numpy() - np.asarray(g)) <= 2 * bound).all(), A.shape
        assert abs(rss[i] - s) <= (m + 4) * U * s, A.shape


@pytest.mark.parametrize("trans", [False, True])
def test_triangular_products_in_and_out_of_place(batch, trans):
    """Both forms give the same bits, and the product's componentwise bound."""
    ops, As, _, B = batch
    print("[bt-passes] trmv", trans, flush=True)
    rng = np.random.default_rng(12)
    L, st = ops.lib(), ops.stream(B.dev)
    Ms = [np.triu(rng.standard_normal((A.shape[1], A.shape[1]))) for A in As]
    # what lies outside the triangle is not read
    up = torch.from_numpy(np.concatenate([(M + np.tril(np.full(M.shape, np.nan), -1)).ravel() for M in Ms])).to(B.dev)
    lo = torch.from_numpy(np.concatenate([(M.T + np.triu(np.full(M.shape, np.nan), 1)).ravel() for M in Ms])).to(B.dev)
    y = torch.full_like(B.t, float("nan"))
    ops.check(L.pamd_bt_trmv_to(B.P, ops._p(B.desc), int(trans), ops._p(up), ops._p(lo), ops._p(B.t), ops._p(y), st),
              "pamd_bt_trmv_to")
    v = B.t.clone()
    ops.check(L.pamd_bt_trmv(B.P, ops._p(B.desc), int(trans), ops._p(up), ops._p(lo), ops._p(v), st), "pamd_bt_trmv")
    assert torch.equal(y, v)
    for i, M in enumerate(Ms):
        T, t = (M.T if trans else M), B.vec(B.t, i).cpu().numpy()
        bound = (M.shape[0] + 2) * U * (np.abs(T) @ np.abs(t))
        assert (np.abs(B.vec(y, i).cpu().numpy() - T @ t) <= 2 * bound).all(), M.shape


@pytest.mark.parametrize("use_graph", [True, False])
def test_launch_shapes_are_timed_on_active_problems(use_graph):
    """Every shape that a fresh solver's first call, and a second call with
    other sizes, puts into its cache was timed with all problems active."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import parla_amd.drivers.batched_ls as bl
    print("[bt-passes] launch shapes", use_graph, flush=True)
    solver = bl.BatchedSPO()
    inner, misses = solver._pass, []

    def spy(B, kind):
        if torch.cuda.is_current_stream_capturing():
            known = set(solver.tuner.cache)
            inner(B, kind)
            assert known == set(solver.tuner.cache)
            return
        active, known = bool((B.state[1::4] == 1).all()), set(solver.tuner.cache)
        inner(B, kind)
        misses.extend((kind, key, active) for key in set(solver.tuner.cache) - known)

    solver._pass = spy
    rng = np.random.default_rng(4)
    for shapes in ([(900, 40), (1500, 100), (2000, 200)], [(3000, 300), (700, 30)]):
        As = [rng.standard_normal(s).astype(np.float32) for s in shapes]
        solver(As, [rng.standard_normal(s[0]) for s in shapes], 1e-10, 1, use_graph=use_graph)
    assert {k for k, _, _ in misses} == {"normal", "residual"}
    assert all(active for _, _, active in misses), misses
