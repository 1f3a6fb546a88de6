"""The exact BF16 sketch product in tiles of two row tiles: bit for bit the
integer chunk sums added in FP64 in the documented order, with an odd number of
row tiles (the last tile half empty: 9, and 5 with more than two pieces; one
high below) and an even one."""
import numpy as np
import pytest
import torch

import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [2, 3, 4])
@pytest.mark.parametrize("d,n", [(300, 500), (200, 1000), (600, 400), (1100, 250)])
def test_tall_tiles_exact(P, d, n):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from parla_amd import ops
    m = 32768 - 5
    print("[gpu-ozaki] tall tiles", d, m, n, P, flush=True)
    dpad, ncp, group = ops.ozaki_layout(d, m, n + 1)[1:4]
    chunks = -(-m // 256)
    assert -(-dpad // 256) * (ncp // 64) * -(-chunks // group) >= 1024  # the tall tiles' range
    rng = np.random.default_rng(d + P)
    dev = torch.device("cuda")
    A, b = torch.from_numpy(rng.standard_normal((m, n))).to(dev), torch.from_numpy(rng.standard_normal(m)).to(dev)
    Z = rng.standard_normal((d, m))
    sp = ops.OzakiSplit(A, b, P)
    scale = 2.0 ** -5 / np.sqrt(d)
    out = ops.ozaki_sketch(ops.quantize_q(torch.from_numpy(Z).to(dev)), d, sp, scale)
    Q = torch.from_numpy(np.asarray(orc.quantize_q(Z), dtype=np.float64)).to(dev)
    pieces = [torch.from_numpy(np.asarray(sp.piece(p), dtype=np.float64)[:n + 1, :m].copy()).to(dev) for p in range(P)]
    exps = sp.exps[:, :n + 1]
    total = torch.zeros(d, n + 1, dtype=torch.float64, device=dev)
    for c0 in range(0, chunks, group):
        acc = torch.zeros_like(total)
        for c in range(c0, min(c0 + group, chunks)):
            sl = slice(256 * c, min(256 * (c + 1), m))
            for p in range(P):  # integers below 2^53: exact in any order
                s = Q[:, sl] @ pieces[p][:, sl].t()
                acc += s * torch.ldexp(torch.ones((), dtype=torch.float64, device=dev), (exps[c] - 8 - 9 * p).double())
        total += acc
    assert torch.equal(out[:, :n + 1], scale * total)
