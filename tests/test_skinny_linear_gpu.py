"""Products of few rows at the edges of their tiles, against float64."""
import warnings

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


def test_transforms_modes_and_traces_see_the_product():
    """Few rows, and something around the call that follows torch's own operations."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode

    g = torch.Generator(device="cuda:0").manual_seed(0)
    xs, w, dx = (torch.randn(*s, device="cuda:0", generator=g).bfloat16() for s in ((3, 4, 64), (40, 64), (4, 64)))
    plain = torch.stack([torch.matmul(x, w.t()) for x in xs]).float()
    tol = 2.0 ** -7 * plain.abs().max()                                    # two roundings to bfloat16
    assert ((torch.vmap(linear, in_dims=(0, None))(xs, w).float() - plain).abs() <= tol).all()
    assert ((torch.vmap(linear, in_dims=(None, 0))(xs[0], torch.stack([w, w]))[1].float() - plain[0]).abs() <= tol).all()
    want = torch.matmul(dx, w.t()).float()
    y, dy = torch.func.jvp(lambda x: linear(x, w), (xs[0],), (dx,))
    assert ((y.float() - plain[0]).abs() <= tol).all() and ((dy.float() - want).abs() <= 2.0 ** -7 * want.abs().max()).all()
    with forward_ad.dual_level():
        dy = forward_ad.unpack_dual(linear(forward_ad.make_dual(xs[0], dx), w)).tangent
    assert dy is not None and ((dy.float() - want).abs() <= 2.0 ** -7 * want.abs().max()).all()

    seen = []

    class Listen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Listen():
        linear(xs[0], w)
    assert any("mm" in f for f in seen), seen
    with warnings.catch_warnings():
        warnings.simplefilter("error", torch.jit.TracerWarning)               # (no decision of the rule's is written into the trace)
        traced = torch.jit.trace(lambda x: linear(x, w), (xs[0],), check_trace=False)
    assert ((traced(xs[1]).float() - plain[1]).abs() <= tol).all()
    wp = torch.nn.Parameter(w)
    x = xs[0].clone().requires_grad_()
    linear(x, wp).float().sum().backward()
    assert x.grad is not None and wp.grad is not None
    for dtype in (torch.float16, torch.float32, torch.bfloat16):
        with torch.autocast("cuda", dtype=dtype, enabled=dtype != torch.float32):
            y, want = linear(xs[0], w), torch.matmul(xs[0], w.t())
        assert y.dtype == want.dtype and ((y.float() - want.float()).abs() <= tol).all()
