"""Products of one to four tokens with the row operation in front of them: the bits of the launches they replace."""
import pytest
import torch

from qserve_amd import fused
from qserve_amd.decode import W4A8Linear, residual_add_

pytestmark = pytest.mark.gpu
GROUPS = pytest.mark.parametrize("group", [-1, 128])


def _linear(n, k, group, g, big_scales=False):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lin = W4A8Linear(n, k, group, "cuda", g)
    if big_scales and group != -1:                          # level-2 products that carry into the next byte
        lin.s2_scales[::2, :40] = torch.randint(17, 127, (len(lin.s2_scales[::2]), 40), dtype=torch.int8, device="cuda", generator=g)
    return lin


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed) if torch.cuda.is_available() else None


def _groups(lin):
    return {} if lin.group_size == -1 else dict(zeros=lin.s2_zeros, scales_i8=lin.s2_scales)


def _gemm(lin, x, scale, total):
    out = torch.empty((x.size(0), lin.n), dtype=torch.float16, device="cuda")
    lin(x, scale, total, out)
    return out


def _sums(lin, x):
    """The int32 sums by torch's own integers (float64 products of whole numbers below 2^53)."""
    one = torch.ones(x.size(0), dtype=torch.float16, device="cuda")
    from qserve_backend import qgemm_w4a8_per_chn as chn, qgemm_w4a8_per_group as grp
    acc = torch.empty((x.size(0), lin.n), dtype=torch.int32, device="cuda")
    if lin.group_size == -1:
        chn.gemm_forward_acc(x, lin.qweight, acc)
    else:
        grp.gemm_forward_acc(x, lin.qweight, lin.s2_zeros, lin.s2_scales, acc)
    return acc


# waves with no stage, with one, with a part of their loads; the widest slices; carries
@GROUPS
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N, K, ks", [(64, 128, 1), (64, 256, 2), (192, 640, 1), (4096, 4096, 2), (128, 4096, 4), (64, 11008, 4), (192, 3840, 1), (64, 14336, 4), (64, 4096, 1)])
def test_planes_of_few_rows(group, M, N, K, ks):
    g = _gen(N + K + M)
    if group != -1 and K % (128 * ks):
        ks //= 2
    if group != -1 and K // ks > 4096:
        pytest.skip("slices of more than 4096")
    lin = _linear(N, K, group, g, big_scales=K > 1000)
    assert fused.rows_ok(M, N, K, ks, group != -1)
    x = torch.randint(-128, 128, (M, K), dtype=torch.int8, device="cuda", generator=g)
    planes = torch.full((ks, M, N), 7, dtype=torch.int32, device="cuda")
    fused.rows_planes(x, lin.qweight, planes, **_groups(lin))
    assert torch.equal(planes.sum(0, dtype=torch.int32), _sums(lin, x))


def _norm_operands(g, M, K, slices, group):
    f16 = lambda *s, scale=1.0: (torch.randn(*s, device="cuda", generator=g) * scale).half()                                  # noqa: E731
    planes = torch.randint(-40000, 40000, (slices, M, K), dtype=torch.int32, device="cuda", generator=g)
    return dict(hidden=f16(M, K), planes=planes, plane_wscales=f16(K, scale=0.002).abs(), plane_ascales=f16(M, scale=0.02).abs(),
                plane_wszs=f16(K, scale=0.01) if group == -1 else None, plane_asums=f16(M, scale=3.0) if group == -1 else None, weight=f16(K).abs(), epsilon=1e-5)


@GROUPS
@pytest.mark.parametrize("slices", [2, 4])
@pytest.mark.parametrize("M, N, silu", [(1, 6144, False), (2, 64, False), (3, 192, False), (4, 4096, False), (1, 28672, True), (2, 128, True), (4, 22016, True)])
def test_norm_in_front_of_a_product(group, slices, M, N, silu):
    K, g = 4096, _gen(N + M)
    lin, o = _linear(N, K, group, g), _norm_operands(g, M, K, slices, group) if torch.cuda.is_available() else None
    q, sc, total = torch.empty((M, K), dtype=torch.int8, device="cuda"), *(torch.empty(M, dtype=torch.float16, device="cuda") for _ in range(2))
    h = o["hidden"].clone()
    fused.add_residual_rms_norm_general_planes(q, h, o["planes"], o["plane_wscales"], o["plane_ascales"], o["weight"], sc, o["epsilon"], w_szs=o["plane_wszs"],
                                               a_ssums=o["plane_asums"], input_sum=total if group == -1 else None)
    if silu:
        ref, tmp = torch.empty((M, N // 2), dtype=torch.float16, device="cuda"), torch.empty((M, N), dtype=torch.float16, device="cuda")
        lin.silu_mul(q, sc, total, ref, tmp)
    else:
        ref = _gemm(lin, q, sc, total)
    out, moved = torch.full_like(ref, float("nan")), torch.empty_like(h)
    before = o["hidden"].clone()
    fused.norm_rows(out, hidden_out=moved, kernel=lin.qweight, wscales=lin.s1_scales, w_szs=lin.s1_szeros if group == -1 else None, silu_mul=silu, **_groups(lin), **o)
    assert torch.equal(out, ref) and torch.equal(moved, h) and torch.equal(o["hidden"], before)


@GROUPS
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N, K, ks", [(4096, 14336, 4), (64, 11008, 4), (64, 8704, 4), (64, 16384, 4), (4096, 4096, 2), (64, 4096, 4), (64, 2304, 1), (128, 3840, 2)])
def test_quantiser_in_front_of_planes(group, M, N, K, ks):
    g = _gen(K + M)
    if group != -1 and K % (128 * ks):
        ks = 2
    if not fused.rows_ok(M, N, K, ks, group != -1):
        pytest.skip("slices of more than 4096")
    lin = _linear(N, K, group, g)
    act = (torch.randn(M, K, device="cuda", generator=g) * torch.rand(M, 1, device="cuda", generator=g)).half()
    from qserve_backend import fused_kernels
    q, (sc, total, sc2, total2) = torch.empty((M, K), dtype=torch.int8, device="cuda"), (torch.empty(M, dtype=torch.float16, device="cuda") for _ in range(4))
    if group == -1:
        fused_kernels.invoke_quant_fuse_sum(q, act, total, sc)
    else:
        fused_kernels.invoke_quant(q, act, sc)
    planes = torch.empty((ks, M, N), dtype=torch.int32, device="cuda")
    fused.quant_rows_planes(planes, act, sc2, lin.qweight, input_sum=total2 if group == -1 else None, **_groups(lin))
    assert torch.equal(planes.sum(0, dtype=torch.int32), _sums(lin, q)) and torch.equal(sc, sc2)
    assert group != -1 or torch.equal(total, total2)


@GROUPS
@pytest.mark.parametrize("slices", [1, 2, 4])
@pytest.mark.parametrize("M, K", [(1, 4096), (64, 4096), (5, 2048), (3, 264)])
def test_norm_behind_the_last_planes(group, slices, M, K):
    g = _gen(M)
    if g is None:
        pytest.skip("no GPU")
    o = _norm_operands(g, M, K, slices, group)
    from qserve_backend import layernorm_ops
    w = dict(w_szs=o["plane_wszs"], a_ssums=o["plane_asums"])
    # the product's result from its planes: the general row operation on a stream of zeros leaves it there
    delta, q, sc = torch.zeros((M, K), dtype=torch.float16, device="cuda"), torch.empty((M, K), dtype=torch.int8, device="cuda"), torch.empty(M, dtype=torch.float16, device="cuda")
    fused.add_residual_rms_norm_general_planes(q, delta, o["planes"], o["plane_wscales"], o["plane_ascales"], o["weight"], sc, 1e-5, **w)
    h, ref = o["hidden"].clone(), torch.empty((M, K), dtype=torch.float16, device="cuda")
    residual_add_(h, delta)
    layernorm_ops.rms_norm(ref, h, o["weight"], 1e-5)
    out = torch.empty_like(ref)
    fused.add_residual_rms_norm_planes(out, o["hidden"], o["hidden"], o["planes"], o["plane_wscales"], o["plane_ascales"], o["weight"], 1e-5, **w)
    assert torch.equal(o["hidden"], h)
    assert torch.equal(out, ref)


def test_a_residual_sum_in_place_is_refused():
    g = _gen(1)
    lin, o = _linear(64, 4096, -1, g), _norm_operands(g, 1, 4096, 2, -1) if g else None
    with pytest.raises(RuntimeError):
        fused.norm_rows(torch.empty((1, 64), dtype=torch.float16, device="cuda"), hidden_out=o["hidden"], kernel=lin.qweight, wscales=lin.s1_scales, w_szs=lin.s1_szeros, **o)
