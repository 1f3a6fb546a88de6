"""The leverage network's gradient at the edges of its work split."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


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


def _check_against_autograd(rows, seed):
    from parla_amd.comps.sketchers.learned import NPARAM, LeverageMLP
    rng = np.random.default_rng(seed)
    theta = (rng.standard_normal(NPARAM) * 0.3).astype(np.float32)
    net = LeverageMLP()
    net.set_theta(theta)
    F = _randn(rows, 16, seed=seed).to(torch.float32)
    t = _randn(rows, seed=seed + 1).to(torch.float32)
    g, loss = net.loss_grad(F, t)
    th = torch.from_numpy(theta).cuda()
    cut = [0, 1024, 1088, 5184, 5248, 5312, 5313]
    W = [th[a:b] for a, b in zip(cut[:-1], cut[1:])]
    for i in (0, 2, 4):
        W[i] = W[i].to(torch.bfloat16)
    P = [p.double().requires_grad_(True) for p in (W[0].reshape(16, 64), W[1], W[2].reshape(64, 64), W[3], W[4], W[5])]
    h = torch.relu(torch.asinh(F.double()) @ P[0] + P[1])
    h = torch.relu(h @ P[2] + P[3])
    ref = torch.mean((h @ P[4] + P[5] - t.double()) ** 2)
    ref.backward()
    ref = ref.detach()
    gr = torch.cat([p.grad.reshape(-1) for p in P])
    # FP32 sums over a row's 64 + 64 units and up to `rows` rows
    assert float((g.double() - gr).norm()) <= 2e-5 * float(gr.norm())
    assert abs(float(loss) - float(ref)) <= 2e-5 * float(ref)


@pytest.mark.parametrize("rows", [15, 16, 17, 127, 128, 129, 32767, 32768, 32769, 40000])
def test_mlp_gradient_edges(ops, rows):
    """The gradient at the edges of a wavefront's 16 rows, a workgroup's 128
    and of one round of the whole grid (32768), against FP64 autograd."""
    print(f"[gpu-mlp-grad] rows={rows}", flush=True)
    sys.stdout.flush()
    _check_against_autograd(rows, rows)


@pytest.mark.parametrize("rows", [524288, 524289, 524288 + 32768 - 15, 1048576 + 17])
def test_mlp_gradient_beyond_one_run(ops, rows):
    """16 rounds of the grid are summed in FP32, the rest goes on in FP64."""
    print(f"[gpu-mlp-grad] rows={rows}", flush=True)
    _check_against_autograd(rows, 7)


def test_mlp_sums_do_not_lose_precision_with_rows(ops):
    """2^24 copies of one row: every entry is the mean of equal terms (a power
    of two of them, so the scaling is exact), and no FP32 sum runs over more
    than 256 rows and eight wavefronts, whatever their number."""
    from parla_amd.comps.sketchers.learned import NPARAM, LeverageMLP
    print("[gpu-mlp-grad] equal rows", flush=True)
    net = LeverageMLP()
    net.set_theta((np.random.default_rng(3).standard_normal(NPARAM) * 0.3).astype(np.float32))
    x = _randn(1, 16, seed=3).to(torch.float32)
    ref, lref = net.loss_grad(x.expand(16, 16).contiguous(), torch.full((16,), 3.0, device="cuda"))
    g, loss = net.loss_grad(x.expand(1 << 24, 16).contiguous(), torch.full((1 << 24,), 3.0, device="cuda"))
    assert int((ref != 0).sum()) > 1000 and bool(((g != 0) == (ref != 0)).all())
    # the runs' additions, and those of the reference's own 16 rows
    tol = (256 + 8 + 16) * 2.0 ** -24
    rel = ((g.double() - ref.double()).abs() / ref.double().abs().clamp_min(1e-30))[ref != 0]
    assert float(rel.max()) <= tol, float(rel.max())
    assert abs(float(loss) - float(lref)) <= tol * float(lref)
