"""Products of few rows at the edges of their tiles, against float64."""
import pytest
import torch

from qserve_amd.layers.ops import linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N, K", [(1, 8), (15, 16), (30, 56), (33, 64), (2047, 72), (2048, 1408), (5120, 136), (6144, 2048), (8194, 264), (16390, 64), (512, 4104)])
def test_few_rows(T, N, K):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    g = torch.Generator(device="cuda:0").manual_seed(T + N)
    wide = torch.randn(T, K + 24, device="cuda:0", generator=g).bfloat16()
    w = torch.randn(N, K, device="cuda:0", generator=g).bfloat16()
    for x in (wide[:, :K].contiguous(), wide[:, 16:16 + K], wide[:, 3:3 + K]):          # (columns of a wider product; a start inside 16 bytes: the vendor's)
        y = linear(x, w).double()
        ref = x.double() @ w.double().T
        # one rounding to bfloat16, float sums of K products (two relative 2^-24 per addition at most, in any order)
        bound = 2.0 ** -8 * ref.abs() + 2.0 ** -22 * K * (x.double().abs() @ w.double().abs().T) + 1e-30
        assert ((y - ref).abs() <= bound).all()


def test_shapes_that_do_not_fit_still_raise():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    x, w = torch.zeros(2, 16, device="cuda:0").bfloat16(), torch.zeros(4, 24, device="cuda:0").bfloat16()
    with pytest.raises(RuntimeError):
        linear(x, w)
