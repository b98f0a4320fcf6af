"""Per-group products over weights widened into scratch (qs_w4a8_per_group_gemm_scratch, ..._silu_mul_scratch) against the plain entries: the same bits."""
import pytest
import torch

from qserve_amd._lib import check, lib

pytestmark = pytest.mark.gpu

# tokens: one more than whole tiles, a half and a quarter tile left, a last round of tiles cut into two and four parts and not at all; k: one step, two, an odd number
SHAPES = [(300, 22016, 1024), (1025, 16384, 256), (1280, 32768, 128), (1409, 12288, 384), (2049, 11008, 384), (2600, 4096, 1152), (4200, 8192, 512), (5331, 4096, 1024),
          (5331, 16384, 256)]


def _problem(M, N, K, dev, wild):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    lo, hi = (-128, 128) if wild else (3, 10)                              # wild: level-2 products that wrap and carry
    s8 = torch.randint(lo, hi, (K // 128, N), dtype=torch.int8, device=dev, generator=g)
    z8 = torch.randint(-128, 128, (K // 128, N), dtype=torch.int8, device=dev, generator=g) if wild else (-(8 * s8.int())).to(torch.int8)
    return (torch.randint(-128, 128, (M, K), dtype=torch.int8, device=dev, generator=g),
            torch.randint(-128, 128, (N, K // 2), dtype=torch.int8, device=dev, generator=g), z8, s8,
            ((torch.rand(N, device=dev, generator=g) + 0.5) * 2e-3).half(), ((torch.rand(M, device=dev, generator=g) + 0.5) * 1e-2).half())


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("wild", [False, True])
def test_bits_of_the_plain_entries(gpu, M, N, K, wild):
    ops = _problem(M, N, K, gpu, wild)
    p, st = [t.data_ptr() for t in ops], torch.cuda.current_stream().cuda_stream
    need = lib.qs_w4a8_per_group_scratch_bytes(M, N, K)
    assert need == N * K
    scratch = torch.empty(need, dtype=torch.uint8, device=gpu)
    a, b = (torch.full((M + 1, N), 7.0, dtype=torch.float16, device=gpu) for _ in range(2))
    check(lib.qs_w4a8_per_group_gemm(*p, a.data_ptr(), M, N, K, st), "plain")
    check(lib.qs_w4a8_per_group_gemm_scratch(*p, b.data_ptr(), M, N, K, scratch.data_ptr(), need, st), "scratch")
    assert torch.equal(a.view(torch.int16), b.view(torch.int16)) and bool((b[M] == 7.0).all())
    tmp = torch.empty((M, N), dtype=torch.float16, device=gpu)
    a, b = (torch.full((M + 1, N // 2), 7.0, dtype=torch.float16, device=gpu) for _ in range(2))
    check(lib.qs_w4a8_per_group_gemm_silu_mul(*p, a.data_ptr(), tmp.data_ptr(), M, N, K, st), "plain")
    check(lib.qs_w4a8_per_group_gemm_silu_mul_scratch(*p, b.data_ptr(), tmp.data_ptr(), M, N, K, scratch.data_ptr(), need, st), "scratch")
    assert torch.equal(a.view(torch.int16), b.view(torch.int16)) and bool((b[M] == 7.0).all())


def test_what_does_not_fit_is_the_plain_entry(gpu):
    M, N, K = 1300, 4096, 1024
    ops, st = _problem(M, N, K, gpu, False), torch.cuda.current_stream().cuda_stream
    p = [t.data_ptr() for t in ops]
    want = torch.empty((M, N), dtype=torch.float16, device=gpu)
    check(lib.qs_w4a8_per_group_gemm(*p, want.data_ptr(), M, N, K, st), "plain")
    scratch = torch.zeros(N * K + 16, dtype=torch.uint8, device=gpu)
    for at, size in ((scratch.data_ptr(), N * K - 1), (scratch.data_ptr() + 8, N * K), (0, 0)):      # too little, off 16 bytes, none
        out = torch.zeros((M, N), dtype=torch.float16, device=gpu)
        check(lib.qs_w4a8_per_group_gemm_scratch(*p, out.data_ptr(), M, N, K, at, size, st), "scratch")
        assert torch.equal(out, want) and not bool(scratch.any())
    for shape in ((256, 22016, 1024), (1024, N, K), (M, 4160, K), (M, N, 1056), (1 << 20, N, 1 << 13), (1152, 12288, 4096), (M, 512, 4096)):
        assert lib.qs_w4a8_per_group_scratch_bytes(*shape) == 0


def test_public_calls_under_capture_and_beside_other_streams(gpu):
    import qserve_backend.qgemm_w4a8_per_group as op
    from qserve_amd import fused
    M, N, K = 1500, 4096, 1024
    X, W, z8, s8, ws, sa = _problem(M, N, K, gpu, False)
    p, st = [t.data_ptr() for t in (X, W, z8, s8, ws, sa)], torch.cuda.current_stream().cuda_stream
    want, act = torch.empty((M, N), dtype=torch.float16, device=gpu), torch.empty((M, N // 2), dtype=torch.float16, device=gpu)
    tmp = torch.empty_like(want)
    check(lib.qs_w4a8_per_group_gemm(*p, want.data_ptr(), M, N, K, st), "plain")
    check(lib.qs_w4a8_per_group_gemm_silu_mul(*p, act.data_ptr(), tmp.data_ptr(), M, N, K, st), "plain")
    outs = [(torch.zeros_like(want), torch.zeros_like(act)) for _ in range(3)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    for _ in range(3):
        for s, (o, a) in zip(streams, outs):
            with torch.cuda.stream(s):
                op.gemm_forward_cuda(X, W, z8, s8, ws, sa, o)
                fused.gemm_silu_and_mul_per_group(X, W, z8, s8, ws, sa, a)
    torch.cuda.synchronize()
    o, a = outs[2]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op.gemm_forward_cuda(X, W, z8, s8, ws, sa, o)
        fused.gemm_silu_and_mul_per_group(X, W, z8, s8, ws, sa, a)
    for _ in range(3):
        o.zero_(), a.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want) and torch.equal(a, act)
    for o, a in outs[:2]:
        assert torch.equal(o, want) and torch.equal(a, act)
