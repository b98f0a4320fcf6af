"""The latent projections' and norms' kernels at the edges of their sizes, against float64."""
import pytest
import torch

from qserve_amd.layers.ops import HipOps, TorchOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _gen(seed):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.Generator(device=DEV).manual_seed(seed)


def _ulp(dtype):
    return 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23


@pytest.mark.parametrize("T, H, K, N", [(1, 1, 32, 32), (3, 2, 96, 64), (16, 16, 512, 128), (17, 3, 128, 512), (32, 2, 256, 160), (33, 5, 1024, 32),
                                        (63, 2, 160, 96), (64, 16, 768, 64)])
def test_one_product_per_head(T, H, K, N):
    g = _gen(T)
    x, w = torch.randn(T, H, K, device=DEV, generator=g).bfloat16(), torch.randn(H, K, N, device=DEV, generator=g).bfloat16()
    y = HipOps(torch.bfloat16).head_products(x, w).double().view(T, H, N)
    ref = torch.einsum("thk,hkn->thn", x.double().cpu(), w.double().cpu()).to(DEV)
    size = torch.einsum("thk,hkn->thn", x.double().abs().cpu(), w.double().abs().cpu()).to(DEV)
    # one rounding to bfloat16, float sums of K products (two relative 2^-24 per addition at most, in any order)
    assert ((y - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -22 * K * size + 1e-30).all()


@pytest.mark.parametrize("T, H, K, N, off", [(1, 1, 32, 32, 0), (17, 3, 128, 160, 2), (64, 16, 512, 128, 1344), (33, 2, 96, 64, 1), (70, 2, 64, 32, 2)])
def test_gated_product_per_head(T, H, K, N, off):
    """The gate a column slice: on two elements (inside the product), on an odd one and beyond 64 rows (a launch of its own, one rounding more)."""
    g = _gen(T)
    x, w = torch.randn(T, H, K, device=DEV, generator=g).bfloat16(), torch.randn(H, K, N, device=DEV, generator=g).bfloat16()
    gate = (torch.randn(T, off + H * N + (off & 1), device=DEV, generator=g) * 3).bfloat16()[:, off:off + H * N]
    y = HipOps(torch.bfloat16).head_products(x, w, gate).double()
    xc, wc, s = x.double().cpu(), w.double().cpu(), torch.sigmoid(gate.double()).cpu()
    ref, size = (torch.einsum("thk,hkn->thn", a, b).reshape(T, -1) * s for a, b in ((xc, wc), (xc.abs(), wc.abs())))
    assert ((y.cpu() - ref).abs() <= (2 if off & 1 or T > 64 else 1) * 2.0 ** -8 * ref.abs() * 1.01 + 2.0 ** -22 * K * size + 1e-30).all()


@pytest.mark.parametrize("T, H, dim, rot_dim, rot_n, rank", [(1, 1, 32, 0, 0, 32), (16, 16, 128, 64, 64, 512), (17, 2, 64, 8, 4, 96), (33, 3, 96, 40, 38, 64),
                                                             (64, 16, 128, 64, 32, 256), (65, 16, 128, 64, 64, 512), (70, 2, 20, 12, 8, 24),
                                                             (5, 3, 33, 7, 2, 31)])
def test_latent_query(T, H, dim, rot_dim, rot_n, rank):
    """Product and rotation in one, the four-column kernel behind the batched product, and the plain one for sizes that are no multiple of four."""
    g = _gen(T)
    q, w = torch.randn(T, H * (dim + rot_dim), device=DEV, generator=g).bfloat16(), torch.randn(H, dim, rank, device=DEV, generator=g).bfloat16()
    pos = torch.randint(0, 50, (T,), device=DEV, generator=g, dtype=torch.int32)
    a = torch.rand(50, max(rot_n // 2, 1), device=DEV, generator=g) * 6.28
    rope = torch.stack([a.cos(), a.sin()], 1).contiguous() if rot_n else None
    qf = HipOps(torch.bfloat16).latent_queries(q, w, rope, pos, 0.125, H, dim, rot_dim, rot_n, rank)
    absorbed = torch.einsum("thk,hkn->htn", q.view(T, H, -1)[..., :dim].double().cpu(), w.double().cpu()).to(DEV)
    size = torch.einsum("thk,hkn->thn", q.view(T, H, -1)[..., :dim].double().abs().cpu(), w.double().abs().cpu()).to(DEV)
    ref = TorchOps(torch.float32).latent_query(q, absorbed, rope, pos, 0.125, H, dim, rot_dim, rot_n, rank).double()
    # the absorbed part rounded to bfloat16 once at most; the rotated part two float products of values below 2^3 and their sum
    bound = torch.cat([2.0 ** -8 * absorbed.transpose(0, 1).abs() + 2.0 ** -22 * dim * size, torch.full((T, H, rot_dim), 2.0 ** -19, device=DEV).double()], -1)
    assert ((qf.double() - ref).abs() <= 0.125 * bound + 1e-30).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T, D", [(1, 4), (3, 6), (2, 1020), (64, 1024), (5, 1028), (65, 2048), (7, 2052), (3, 4096), (3, 4100)])
def test_layer_norms(T, D, dtype):
    g = _gen(T + D)
    x0 = torch.randn(T, D, device=DEV, generator=g)
    y, w = (torch.randn(T, D, device=DEV, generator=g) * 2 + 0.5).to(dtype), torch.randn(D, device=DEV, generator=g).to(dtype)
    rows = torch.randperm(T, device=DEV, generator=g).to(torch.int32)[:max(1, T // 2)]

    def normed(v):
        v = v.double()
        c = v - v.mean(-1, keepdim=True)
        return c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-5) * w.double()

    ops, x = HipOps(dtype), x0.clone()
    h = ops.add_layer_norm(x, y, w, 1e-5)
    ref = x0.double() + normed(y)
    # float statistics of D values (relative 2^-24 per addition in each of the two sums), a few float roundings behind them
    bound = (2.0 ** -24 * D + 2.0 ** -20) * (x0.double().abs() + normed(y).abs() + w.double().abs())
    assert ((x.double() - ref).abs() <= bound).all() and ((h.double() - x.double()).abs() <= _ulp(dtype) * x.double().abs()).all()
    out = ops.layer_norm_rows(x0, rows, w, 1e-5).double()
    ref = normed(x0)[rows.long()]
    assert ((out - ref).abs() <= (2.0 ** -24 * D + 2.0 ** -20) * (ref.abs() + w.double().abs()) + _ulp(dtype) * ref.abs()).all()
