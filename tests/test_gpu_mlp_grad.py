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


@pytest.mark.parametrize("rows", [15, 16, 17, 127, 128, 129, 32767, 32768, 32769, 40000])
def test_mlp_gradient_edges(ops, rows):
    """The gradient at the edges of a wavefront's 16 rows, a workgroup's 128
    and of one round of the whole grid (32768), against FP64 autograd."""
    print(f"[gpu-mlp-grad] rows={rows}", flush=True)
    sys.stdout.flush()
    from parla_amd.comps.sketchers.learned import NPARAM, LeverageMLP
    rng = np.random.default_rng(rows)
    theta = (rng.standard_normal(NPARAM) * 0.3).astype(np.float32)
    net = LeverageMLP()
    net.set_theta(theta)
    F = _randn(rows, 16, seed=rows).to(torch.float32)
    t = _randn(rows, seed=rows + 1).to(torch.float32)
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
