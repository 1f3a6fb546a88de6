"""Timed cases of the library's main paths, through its public entry points.

Each case is one call that a user of the package makes: a least-squares solve
(``SPO``, ``SPOMixed``, ``BatchedSPO``), a low-rank decomposition (``QB1``,
``SVD1``, ``EVD1``), the products of a ``SplitOperator`` or a training step of
``LeverageMLP``.  ``listed`` gives fixed cases, ``draw`` further ones of the
same ranges, ``prepare`` the data a program holds before the call, ``run`` the
call, ``work`` what it cannot do without, ``exact`` the result in plain FP64.
"""
import math

import numpy as np
import torch

import parla_amd as pa
from parla_amd.comps.sketchers.learned import NPARAM, LeverageMLP
from parla_amd.drivers.batched_ls import BatchedSPO

F64 = torch.float64


def listed():
    return [
        # the smallest solves: a regression of the size of the test problems, where launches and host work count
        dict(name="spo_small", kind="spo", m=1000, n=100, sketch="sjlt", cond=1e4, delta=0.0),
        # the plain FP64 least-squares workload (Gaussian sketch, Householder QR, preconditioned LSQR)
        dict(name="spo_gauss", kind="spo", m=20000, n=200, sketch="gauss", cond=1e6, delta=0.0),
        # ridge regression on odd sizes
        dict(name="spo_ridge_odd", kind="spo", m=50021, n=333, sketch="sjlt", cond=1e5, delta=1e-6),
        # a tall problem with the sparse sketch (the shape of the learned-sketch workload, FP64)
        dict(name="spo_tall", kind="spo", m=131072, n=512, sketch="sjlt", cond=1e5, delta=0.0),
        # mixed precision with FP64 refinement: the ordinary and the largest solve
        dict(name="mixed_mid", kind="mixed", m=20000, n=200, cond=1e6),
        dict(name="mixed_large", kind="mixed", m=262144, n=1024, cond=1e6),
        # many small and middle problems in one call
        dict(name="batched", kind="batched", problems=64, m_min=2000, m_max=50000, n_min=32, n_max=512, shapes=4),
        # the low-rank workload: QB with two power iterations, and the SVD behind it on a smaller odd matrix
        dict(name="qb_large", kind="qb", m=8192, n=4096, k=266),
        dict(name="qb_small", kind="qb", m=1000, n=700, k=40),
        dict(name="svd_odd", kind="svd", m=3001, n=2003, k=150, over=10),
        # the power iteration's products with A as BF16 pieces, both directions
        dict(name="split_products", kind="split", m=8192, n=4096, k=266, pieces=2),
        # one training step of the leverage-score network: forward, backward, Adam
        dict(name="mlp_step", kind="mlp", rows=65536),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["spo", "spo", "spo", "mixed", "mixed", "batched", "qb", "qb", "svd", "evd", "split", "mlp"])
    cond = 10.0 ** rng.uniform(1.0, 6.0)
    if kind == "spo":
        n = _log_int(rng, 20, 512)
        return dict(kind=kind, m=_log_int(rng, 8 * n, 131072), n=n, sketch=rng.choice(["sjlt", "gauss"]), cond=cond,
                    delta=rng.choice([0.0, 0.0, 1e-6]))
    if kind == "mixed":
        n = _log_int(rng, 50, 1024)
        return dict(kind=kind, m=_log_int(rng, 16 * n, 262144), n=n, cond=cond)
    if kind == "batched":
        return dict(kind=kind, problems=_log_int(rng, 8, 64), m_min=2000, m_max=_log_int(rng, 8000, 50000), n_min=32,
                    n_max=_log_int(rng, 100, 512), shapes=rng.randrange(10 ** 6))
    if kind == "mlp":
        return dict(kind=kind, rows=_log_int(rng, 1000, 65536))
    m, n = _log_int(rng, 500, 8192), _log_int(rng, 500, 4096)
    if kind == "split":
        return dict(kind=kind, m=m, n=n, k=_log_int(rng, 16, 266), pieces=rng.choice([2, 3]))
    if kind == "evd":
        return dict(kind=kind, m=n, n=n, k=_log_int(rng, 10, min(150, n // 8)), over=10)
    if kind == "svd":
        return dict(kind=kind, m=m, n=n, k=_log_int(rng, 10, min(150, min(m, n) // 8)), over=10)
    return dict(kind=kind, m=m, n=n, k=_log_int(rng, 10, min(266, min(m, n) // 4)))


# --------------------------------------------------------------------------- data

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) + 20260000)
    return g


def _randn(g, *shape, dtype=F64):
    return torch.randn(*shape, dtype=dtype, device="cuda", generator=g)


def _ls_problem(g, m, n, cond, noise=1e-8):
    """A = G diag(s) V^T with Gaussian G (near-orthonormal columns), s geometric from 1 to 1/cond, V orthogonal;
    b = A x + noise N(0, 1)."""
    V = torch.linalg.qr(_randn(g, n, n).cpu())[0].cuda()
    s = torch.logspace(0.0, -math.log10(cond), n, dtype=F64, device="cuda")
    A = _randn(g, m, n) @ ((s / math.sqrt(m))[:, None] * V.t())
    b = A @ _randn(g, n) + noise * _randn(g, m)
    return A, b


def _low_rank(g, m, n, k):
    """Polynomially decaying spectrum over a noise floor: sum_i i^-1 u_i v_i^T (i <= 2 k) + 1e-6 noise."""
    r = min(2 * k, m, n)
    s = torch.arange(1, r + 1, dtype=F64, device="cuda") ** -1.0
    A = (_randn(g, m, r) * (s / math.sqrt(m))) @ (_randn(g, n, r).t() / math.sqrt(n))
    return A + 1e-6 / math.sqrt(m) * _randn(g, m, n)


def _psd(g, n, k):
    r = min(2 * k, n)
    s = torch.arange(1, r + 1, dtype=F64, device="cuda") ** -1.0
    G = _randn(g, n, r) / math.sqrt(n)
    A = (G * s) @ G.t()
    return 0.5 * (A + A.t())


def _batch_shapes(case):
    rng = np.random.default_rng(case["shapes"])
    out = []
    while len(out) < case["problems"]:
        m = int(rng.integers(case["m_min"], case["m_max"] + 1))
        n = int(rng.integers(case["n_min"], case["n_max"] + 1))
        if m >= 8 * n:
            out.append((m, n, 10.0 ** rng.uniform(1.0, 4.0)))
    return out


def _mlp_theta(seed):
    rng = np.random.default_rng(seed)
    return np.concatenate([rng.normal(0, math.sqrt(2.0 / 16), 16 * 64), 0.1 * rng.standard_normal(64),
                           rng.normal(0, math.sqrt(2.0 / 64), 64 * 64), 0.1 * rng.standard_normal(64),
                           rng.normal(0, math.sqrt(1.0 / 64), 64), np.zeros(1)]).astype(np.float32)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "spo":
        A, b = _ls_problem(g, case["m"], case["n"], case["cond"])
        gen = pa.SkOpGA(backend="device") if case["sketch"] == "gauss" else pa.SkOpSJ(8, backend="device")
        return dict(kind=kind, A=A, b=b, alg=pa.SPO(gen, 4), delta=case["delta"], seed=seed)
    if kind == "mixed":
        A, b = _ls_problem(g, case["m"], case["n"], case["cond"])
        return dict(kind=kind, A=A, b=b, alg=pa.SPOMixed(4, backend="device"), seed=seed)
    if kind == "batched":
        probs = [_ls_problem(g, m, n, cond) for m, n, cond in _batch_shapes(case)]
        As = [A.to(torch.float32) for A, _ in probs]
        return dict(kind=kind, As=As, bs=[b for _, b in probs], alg=BatchedSPO(cg_iters=20), seed=seed)
    if kind in ("qb", "svd", "evd"):
        A = _psd(g, case["n"], case["k"]) if kind == "evd" else _low_rank(g, case["m"], case["n"], case["k"])
        qb = pa.QB1(pa.RF1(pa.RS1(pa.SkOpSJ(8, backend="device"), 4, pa.orth, 1)))
        alg = {"qb": qb, "svd": pa.SVD1(qb), "evd": pa.EVD1(qb)}[kind]
        return dict(kind=kind, A=A, alg=alg, k=case["k"], over=case.get("over", 0), seed=seed)
    if kind == "split":
        S = torch.linalg.qr(_randn(g, case["n"], case["k"]).cpu())[0].cuda().contiguous()
        Q = torch.linalg.qr(_randn(g, case["m"], case["k"]).cpu())[0].cuda().contiguous()
        return dict(kind=kind, A=_low_rank(g, case["m"], case["n"], case["k"]), S=S, Q=Q, pieces=case["pieces"])
    net = LeverageMLP(seed=0)
    net.set_theta(_mlp_theta(seed))
    F = _randn(g, case["rows"], 16, dtype=torch.float32)
    t = _randn(g, case["rows"], dtype=torch.float32)
    return dict(kind=kind, net=net, F=F, t=t)


def run(state):
    kind = state["kind"]
    if kind == "spo":
        x, _ = state["alg"](state["A"], state["b"], state["delta"], 1e-12, 100, state["seed"], logging=False)
        return x
    if kind == "mixed":
        x, _ = state["alg"](state["A"], state["b"], 0.0, 1e-10, 100, state["seed"], logging=False)
        return x
    if kind == "batched":
        xs, _ = state["alg"](state["As"], state["bs"], 1e-10, state["seed"])
        return xs
    if kind == "qb":
        return state["alg"](state["A"], state["k"], float("nan"), state["seed"])
    if kind in ("svd", "evd"):
        return state["alg"](state["A"], state["k"], float("nan"), state["over"], state["seed"])
    if kind == "split":
        op = pa.SplitOperator(state["A"], state["pieces"])
        return op @ state["S"], op.T @ state["Q"], state["Q"].t() @ op
    g, loss = state["net"].loss_grad(state["F"], state["t"])
    state["net"].adam(g, lr=2e-3)
    return g, loss, state["net"].w


# --------------------------------------------------------------------------- work and reference

def work(case):
    kind = case["kind"]
    if kind in ("spo", "mixed"):
        m, n = case["m"], case["n"]
        d = 4 * n
        sk = 2.0 * 8 * m * n if case.get("sketch") == "sjlt" else 2.0 * d * m * n
        qr = 2.0 * d * n * n - 2.0 * n ** 3 / 3
        # a dozen products with A and A^T in the mixed form's refinement, about thirty in plain LSQR; A once in memory
        passes = 12 if kind == "mixed" else 30
        return dict(bytes=8.0 * (m * n + m + n), flops=sk + qr + passes * 4.0 * m * n)
    if kind == "batched":
        fl = by = 0.0
        for m, n, _ in _batch_shapes(case):
            fl += 16.0 * m * n + 3 * 4.0 * n * n * n + 40 * 4.0 * m * n
            by += 4.0 * m * n + 8.0 * (m + n)
        return dict(bytes=by, flops=fl)
    if kind == "mlp":
        return dict(bytes=4.0 * case["rows"] * 17 + 16.0 * NPARAM, flops=6.0 * 5200 * case["rows"])
    m, n, k = case["m"], case["n"], case["k"] + case.get("over", 0)
    if kind == "split":
        pairs = case["pieces"] * (case["pieces"] + 1) // 2
        return dict(bytes=8.0 * (m * n + 3 * (m + n) * k), flops=3 * pairs * 2.0 * m * n * k)
    passes = 5 * 2.0 * m * n * k + 16.0 * m * n + 3 * 4.0 * (m + n) * k * k
    return dict(bytes=8.0 * (m * n + (m + n) * k), flops=passes + (30.0 * k ** 3 if kind != "qb" else 0.0))


def _lstsq(A, b, delta=0.0):
    """Householder QR solution of min ||A x - b||^2 + delta ||x||^2 with one step of refinement."""
    n = A.shape[1]
    A, b = A.to(F64), b.to(F64)
    if delta > 0:
        A = torch.cat((A, math.sqrt(delta) * torch.eye(n, dtype=F64, device=A.device)))
        b = torch.cat((b, torch.zeros(n, dtype=F64, device=A.device)))
    Q, R = torch.linalg.qr(A)
    x = torch.zeros(n, 1, dtype=F64, device=A.device)
    for _ in range(3):
        r = b[:, None] - A @ x
        x = x + torch.linalg.solve_triangular(R, Q.t() @ r, upper=True)
    return x[:, 0]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("qb", "svd", "evd"):
        return None  # a randomized approximation: its draws are the library's
    st = prepare(case, seed)
    if kind in ("spo", "mixed"):
        return _lstsq(st["A"], st["b"], st.get("delta", 0.0))
    if kind == "batched":
        return [_lstsq(A, b) for A, b in zip(st["As"], st["bs"])]
    if kind == "split":
        A, S, Q = st["A"], st["S"], st["Q"]
        return A @ S, A.t() @ Q, Q.t() @ A
    # gradient of mean (MLP(asinh F) - t)^2 in FP64 with the weights rounded to BF16, as the network stores them
    F, t = st["F"].to(F64), st["t"].to(F64)
    th = torch.from_numpy(_mlp_theta(seed)).cuda()
    cut = [0, 1024, 1088, 5184, 5248, 5312, 5313]
    W1, b1, W2, b2, w3, b3 = (th[a:b] for a, b in zip(cut[:-1], cut[1:]))
    W1, W2, w3 = (w.to(torch.bfloat16).to(F64) for w in (W1, W2, w3))
    P = [p.to(F64).requires_grad_(True) for p in (W1.reshape(16, 64), b1, W2.reshape(64, 64), b2, w3, b3)]
    h = torch.relu(torch.asinh(F) @ P[0] + P[1])
    h = torch.relu(h @ P[2] + P[3])
    loss = torch.mean((h @ P[4] + P[5] - t) ** 2)
    loss.backward()
    return torch.cat([p.grad.reshape(-1) for p in P]), loss.detach(), None
