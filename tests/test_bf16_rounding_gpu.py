"""What leaves a kernel as bfloat16 is the float rounded to nearest even: one value at a time and in pairs, over products with ties, overflows and subnormals."""
import pytest
import torch

from qserve_amd.layers.ops import ExpertRows, make_ops

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.view(torch.int16)


def test_every_square(gpu):
    """8-bit significands squared: 16 bits, every tie among them."""
    x = torch.arange(1 << 16, dtype=torch.int32, device=gpu).to(torch.int16).view(torch.bfloat16)
    x = x[~x.isnan()]
    got = make_ops("hip", torch.bfloat16, gpu).relu_sq(x.clone())
    v = x.float().clamp(min=0.0)
    assert torch.equal(_bits(got), _bits((v * v).bfloat16()))
    nan = make_ops("hip", torch.bfloat16, gpu)
    rows = torch.full((1, 8), float("nan"), dtype=torch.bfloat16, device=gpu)
    one = torch.ones((1, 1), dtype=torch.float32, device=gpu)
    none = torch.zeros((1, 1), dtype=torch.int32, device=gpu)
    assert bool(ExpertRows(nan, rows, none, one, none, rows, 1).dense().isnan().all())


@pytest.mark.parametrize("scale", [1.0, 1e-38, 1e-40, 3e38])
def test_products_in_pairs(gpu, scale):
    g = torch.Generator(device=gpu).manual_seed(5)
    T, D = 257, 1024
    ys = torch.randn((T, D), device=gpu, generator=g).bfloat16()
    ys[0, :4] = torch.tensor([float("inf"), -float("inf"), 0.0, -0.0])
    wt = (torch.randn((T, 1), device=gpu, generator=g) * scale).clamp(-3.4e38, 3.4e38)
    wt[1] = 1.0 + 2.0 ** -8                                                # (a tie for every significand below 128)
    idx, place = torch.zeros((T, 1), dtype=torch.int32, device=gpu), torch.arange(T, dtype=torch.int32, device=gpu)
    got = ExpertRows(make_ops("hip", torch.bfloat16, gpu), ys, place, wt, idx, ys, 1).dense()
    want = (wt * ys.float()).bfloat16()
    same = (_bits(got) == _bits(want)) | (got == want) | (got.isnan() & want.isnan())          # (0 + -0 is 0)
    assert bool(same.all())
