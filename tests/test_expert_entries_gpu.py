"""Entries of the C ABI that take slots sorted by the caller, against float64 (the engine sorts on the device and uses others)."""
import pytest
import torch

from qserve_amd.serving._lib import check, lib

pytestmark = pytest.mark.gpu
ACTS = pytest.mark.parametrize("act, limit", [(0, 0.0), (1, 0.0), (2, 0.0), (3, 1.0)], ids=["none", "relu_sq", "glu", "clamped_glu"])


def _inputs(counts, top, N, K, act, indexed, weighted):
    """Slots sorted by expert (counts of them each), slot s of the list being slot order[s] of the tokens'."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    g = torch.Generator().manual_seed(N + K + len(counts))
    n = sum(counts)
    order = torch.randperm(n, generator=g) if indexed else None
    X = torch.randn((n + top - 1) // top if indexed else n, K, generator=g).bfloat16()
    W = (torch.randn(len(counts), N, K, generator=g) / K ** 0.5).bfloat16()
    wt = torch.rand(n, generator=g) if weighted else None
    rows = X[order // top] if indexed else X
    iw = torch.ones(n) if wt is None else wt[order] if indexed else wt
    z = torch.cat([rows[a:a + c].double() @ W[e].double().T for e, (a, c) in enumerate(zip(torch.tensor([0] + list(counts)).cumsum(0).tolist(), counts))])
    z = z * iw.double()[:, None]
    if act == 1:
        z = torch.relu(z) ** 2
    elif act == 2:
        z = z[:, 0::2] * torch.sigmoid(z[:, 0::2]) * z[:, 1::2]
    elif act == 3:
        p = z[:, 0::2].clamp(max=1.0)
        z = p * torch.sigmoid(1.702 * p) * (z[:, 1::2].clamp(-1.0, 1.0) + 1.0)
    d = lambda t: None if t is None else t.cuda()                                                # noqa: E731
    return d(order), d(X), d(W), d(wt), z, torch.full(z.shape, float("nan"), dtype=torch.bfloat16, device="cuda")


def _close(out, ref, K):
    # one rounding to bfloat16 and a float sum of K products with unit spread, squared or multiplied by a value below 8 at most
    assert ((out.double().cpu() - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -22 * K ** 0.5 * 64).all()


# tiles of up to 128 slots (an empty one among them), rows that do not fill a tile of 256, more tiles than workgroups
@pytest.mark.parametrize("counts, top, N, K", [((1,), 1, 4, 64), ((64, 0, 65, 128), 2, 132, 192), ((129, 7, 300), 3, 260, 128), ((40,) * 90, 4, 1024, 64)])
@pytest.mark.parametrize("indexed, weighted", [(True, False), (True, True), (False, True)])
@ACTS
def test_tiles_that_the_caller_lists(counts, top, N, K, indexed, weighted, act, limit):
    order, X, W, wt, ref, out = _inputs(counts, top, N, K, act, indexed, weighted)
    L, s, tiles, a = lib(), torch.cuda.current_stream().cuda_stream, [], 0
    for e, c in enumerate(counts):
        tiles += [(e, a + o, min(L.qsv_grouped_gemm_tile_slots(), c - o)) for o in range(0, c, L.qsv_grouped_gemm_tile_slots())] or [(e, a, 0)]
        a += c
    tiles = torch.tensor(tiles, dtype=torch.int32, device="cuda")
    check(L.qsv_grouped_gemm(out.data_ptr(), X.data_ptr(), None if order is None else order.data_ptr(), top, W.data_ptr(), tiles.data_ptr(), tiles.size(0),
                             N, K, act, limit, None if wt is None else wt.data_ptr(), s), "grouped_gemm")
    _close(out, ref, K)
    assert K % L.qsv_grouped_gemm_k_step() == 0


# runs of 16, 32 and more slots, empty ones, rows that do not fill 32, the last stage of the reduction part-empty
@pytest.mark.parametrize("counts, top, N, K", [((1,), 1, 2, 8), ((16, 0, 17), 3, 34, 72), ((33, 2, 70, 0), 4, 66, 4104), ((5,) * 40, 2, 128, 200)])
@pytest.mark.parametrize("indexed, weighted", [(True, False), (True, True), (False, True)])
@ACTS
def test_runs_that_the_caller_sorted(counts, top, N, K, indexed, weighted, act, limit):
    order, X, W, wt, ref, out = _inputs(counts, top, N, K, act, indexed, weighted)
    offsets = torch.tensor([0] + list(counts)).cumsum(0).cuda()
    check(lib().qsv_expert_rows(out.data_ptr(), X.data_ptr(), None if order is None else order.data_ptr(), top, W.data_ptr(), offsets.data_ptr(), len(counts), N, K,
                                act, limit, None if wt is None else wt.data_ptr(), torch.cuda.current_stream().cuda_stream), "expert_rows")
    _close(out, ref, K)


# As many slots as half of the experts (workgroups by slot) and one more (by expert), against the same slots among enough without an expert to be done by expert
# whatever their number; an expert twice, slots without one, rows that do not fill 32, the shared expert's rows fewer and more than the others'
@pytest.mark.parametrize("n, E, top, N, K, shared", [(1, 1030, 1, 34, 64, 0), (8, 16, 4, 1066, 136, 1100), (9, 17, 3, 1066, 136, 700), (9, 18, 3, 1066, 136, 700), (40, 80, 8, 256, 1032, 0)])
@ACTS
def test_few_slots(n, E, top, N, K, shared, act, limit):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    g = torch.Generator().manual_seed(n + E)
    idx = torch.randint(0, E, (n,), generator=g, dtype=torch.int32)
    if n > 4:
        idx[[1, 4]] = E - 1
        idx[2], idx[3] = -1, E
    T = (n + top - 1) // top
    X = torch.randn(3 * E, K, generator=g).bfloat16().cuda()
    W, sW = ((torch.randn(e, r, K, generator=g) / K ** 0.5).bfloat16().cuda() for e, r in ((E, N), (1, max(shared, 1))))
    out_of = lambda rows, r: torch.full((rows, r // 2 if act >= 2 else r), float("nan"), dtype=torch.bfloat16, device="cuda")          # noqa: E731

    def run(idx):
        out, own, s = out_of(len(idx), N), out_of(3 * E, shared), torch.cuda.current_stream().cuda_stream
        args = out.data_ptr(), 0, X.data_ptr(), top, W.data_ptr(), idx.data_ptr(), len(idx), E, N, K, act, limit, None
        if shared:
            check(lib().qsv_expert_slots_shared(*args, own.data_ptr(), X.data_ptr(), sW.data_ptr(), T, shared, K, s), "expert_slots_shared")
        else:
            check(lib().qsv_expert_slots(*args, s), "expert_slots")
        return out[:n], own[:T]

    few, few_shared = run(idx.cuda())
    by_expert, shared_too = run(torch.cat([idx, torch.full((2 * E,), -1, dtype=torch.int32)]).cuda())
    there = ((idx >= 0) & (idx < E)).cuda()
    assert not few[there].isnan().any() and few[~there].isnan().all()
    assert torch.equal(few[there], by_expert[there]) and torch.equal(few_shared, shared_too)


# Gates over their whole range, products that are sums of one term: the units of a prompt's kernel are a step's, and within a rounding of the exact ones
@pytest.mark.parametrize("act, limit", [(2, 0.0), (3, 7.0), (3, 100.0)])
def test_units_over_the_range_of_their_gates(act, limit):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    g = torch.arange(0x3A80, 0x42C9, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)          # 2^-10 .. 100, every bfloat16
    g = torch.cat([g, -g])
    X = torch.zeros(len(g), 64, dtype=torch.bfloat16)
    X[:, 0], X[:, 1], X[:, 2] = g, 1.0, -0.40625
    W = torch.zeros(1, 4, 64, dtype=torch.bfloat16)
    W[0, 0, 0] = W[0, 1, 1] = W[0, 2, 0] = W[0, 3, 2] = 1.0                                          # (gate, 1), (gate, -0.40625)
    X, W = X.cuda(), W.cuda()
    L, s, n = lib(), torch.cuda.current_stream().cuda_stream, len(g)
    listed, sorted_, rows = (torch.full((n, 2), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(3))
    tiles = torch.tensor([(0, o, min(L.qsv_grouped_gemm_tile_slots(), n - o)) for o in range(0, n, L.qsv_grouped_gemm_tile_slots())], dtype=torch.int32, device="cuda")
    check(L.qsv_grouped_gemm(listed.data_ptr(), X.data_ptr(), None, 1, W.data_ptr(), tiles.data_ptr(), tiles.size(0), 4, 64, act, limit, None, s), "grouped_gemm")
    order, offsets = torch.arange(n, dtype=torch.int32, device="cuda"), torch.tensor([0, n], dtype=torch.int32, device="cuda")
    check(L.qsv_grouped_gemm_sorted(sorted_.data_ptr(), X.data_ptr(), order.data_ptr(), 1, W.data_ptr(), offsets.data_ptr(), 1, 4, 64, act, limit, None, s), "sorted")
    check(L.qsv_expert_rows(rows.data_ptr(), X.data_ptr(), None, 1, W.data_ptr(), offsets.long().data_ptr(), 1, 4, 64, act, limit, None, s), "expert_rows")
    assert torch.equal(listed.view(torch.int16), rows.view(torch.int16)) and torch.equal(sorted_.view(torch.int16), rows.view(torch.int16))
    z, u = g.double()[:, None], torch.tensor([1.0, -0.40625], dtype=torch.float64)
    if act == 3:
        z, u = z.clamp(max=limit), u.clamp(-limit, limit) + 1.0
    c = 1.702 if act == 3 else 1.0
    want, near = z * torch.sigmoid(c * z) * u, (c * z > -87.0).expand(-1, 2)                          # (below, 1 + exp leaves a float's range)
    # one rounding to the 8 bits of a bfloat16 (2^-8); before it the exponential, a sum, a quotient and a product: 2^-24 each, the exponent's own rounding (1.702 g) times |c z|
    bound = want.abs() * (2.0 ** -8 + (4 + c * z.abs()) * 2.0 ** -23)
    assert ((listed.double().cpu() - want).abs() <= bound)[near].all()
