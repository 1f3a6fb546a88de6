"""Both orientations' BF16 pieces from one read: the bytes of the two separate splits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [2, 3])
@pytest.mark.parametrize("rows,cols,ld", [(1, 1, 1), (63, 65, 65), (64, 128, 128), (129, 64, 80), (37, 200, 203),
                                          (300, 127, 127), (515, 1030, 1031)])
def test_same_bytes_as_separate_splits(P, rows, cols, ld):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from parla_amd import ops
    print("[gpu-split] both", P, rows, cols, ld, flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(rows + cols)
    X = torch.randn(rows, ld, dtype=torch.float64, device="cuda", generator=g)[:, :cols]
    X[0, 0] = 0.0
    L, Lt = ops.split_both_bf16(X, P)
    for got, want in ((L, ops.split_bf16(X, P)), (Lt, ops.split_bf16(X, P, transpose=True))):
        assert (got.rows, got.K) == (want.rows, want.K)
        assert torch.equal(got.pieces.view(torch.int16), want.pieces.view(torch.int16))
