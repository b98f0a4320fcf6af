"""Decode-shape products over every length of a group's share of the reduction (shorter than the ring, as long, one or more rounds past it, odd and even), against
the integer products of the oracle's operands; per group with level-2 scales at and past the largest whose byte products cannot carry (17)."""
import numpy as np
import pytest
import torch

from oracle import w4a8
from qserve_amd._lib import check, lib

pytestmark = pytest.mark.gpu

# 16-token tiles, 64-channel units and K slices of a workgroup; one stage is 64 k, and 8 / units groups share the stages
GEOMETRIES = [(1, 1, 1), (2, 1, 1), (4, 1, 1), (2, 2, 1), (4, 2, 1), (8, 2, 1), (4, 4, 1), (1, 1, 2), (4, 2, 2)]
STAGES = [1, 2, 3, 4, 5, 6, 7, 8, 11]


def _acc(mode, A, W, Z, S, M, N, K, geometry):
    tiles, units, slices = geometry
    acc = torch.full((M + 1, N), -7, dtype=torch.int32, device=A.device)
    st = torch.cuda.current_stream().cuda_stream
    lib.qs_set_gemm_variant(4100 + 100 * (slices - 1) + 10 * tiles + units)
    try:
        if mode:
            check(lib.qs_w4a8_per_group_gemm_acc(A.data_ptr(), W.data_ptr(), Z.data_ptr(), S.data_ptr(), acc.data_ptr(), M, N, K, st), "acc")
        else:
            check(lib.qs_w4a8_per_chn_gemm_acc(A.data_ptr(), W.data_ptr(), acc.data_ptr(), M, N, K, st), "acc")
    finally:
        lib.qs_set_gemm_variant(-1)
    assert bool((acc[M] == -7).all())
    return acc[:M].cpu().numpy()


@pytest.mark.parametrize("stages", STAGES)
@pytest.mark.parametrize("geometry", GEOMETRIES)
def test_every_number_of_rounds(gpu, geometry, stages):
    tiles, units, slices = geometry
    M, N, K = 16 * tiles - 3, 256, 64 * (8 // units) * slices * stages
    rng = np.random.default_rng(100 * tiles + 10 * units + stages)
    A = rng.integers(-127, 128, (M, K), dtype=np.int8)
    W = rng.integers(-128, 128, (N, K // 2), dtype=np.int8)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)                       # noqa: E731
    a, w = dev(A), dev(W)
    plain = A.astype(np.int64) @ w4a8.unpack_qweight(W).astype(np.int64).T
    assert np.array_equal(_acc(0, a, w, None, None, M, N, K, geometry), plain)
    if K % 128:
        return
    G = K // 128
    Z = rng.integers(-128, 128, (G, N), dtype=np.int8)
    S = rng.integers(1, 18, (G, N), dtype=np.int8)
    S[:, 64:128] = 17
    over, negative = S.copy(), S.copy()
    over[rng.integers(G), rng.integers(N)] = 18                                             # one wave leaves the cheap form in one group
    negative[rng.integers(G), rng.integers(N)] = -1
    for s in (S, over, negative, rng.integers(-128, 128, (G, N), dtype=np.int8)):
        want = w4a8.gemm_per_group_acc(A, W, Z, s)
        assert np.array_equal(_acc(1, a, w, dev(Z), dev(s), M, N, K, geometry), want)


# stages that the groups do not share out evenly: the last round of some groups is empty, slices differ by a pair of stages
@pytest.mark.parametrize("geometry, K", [((1, 1, 1), 3712), ((2, 1, 1), 3840), ((4, 1, 1), 3968), ((2, 2, 1), 1920), ((4, 2, 1), 3712), ((1, 1, 2), 7808),
                                         ((4, 2, 2), 3712), ((4, 4, 2), 2176), ((1, 1, 4), 11008), ((2, 1, 4), 11008), ((2, 2, 4), 11008), ((4, 1, 3), 11008)])
def test_groups_without_a_stage_in_the_last_round(gpu, geometry, K):
    tiles, units, slices = geometry
    M, N = 16 * tiles - 3, 256
    rng = np.random.default_rng(K + tiles)
    A, W = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-128, 128, (N, K // 2), dtype=np.int8)
    Z, S = rng.integers(-128, 128, (K // 128, N), dtype=np.int8), rng.integers(1, 17, (K // 128, N), dtype=np.int8)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)                       # noqa: E731
    a, w, z, s = dev(A), dev(W), dev(Z), dev(S)
    plain, group = A.astype(np.int64) @ w4a8.unpack_qweight(W).astype(np.int64).T, w4a8.gemm_per_group_acc(A, W, Z, S)
    for _ in range(2):                                                                      # (the second finds what the first left in the slices' workspace)
        assert np.array_equal(_acc(0, a, w, None, None, M, N, K, geometry), plain)
        assert np.array_equal(_acc(1, a, w, z, s, M, N, K, geometry), group)
    if slices in (2, 4):                                                                    # as planes: every slice its own sum
        st = torch.cuda.current_stream().cuda_stream
        lib.qs_set_gemm_variant(4600 + 100 * (slices - 1) + 10 * tiles + units)
        try:
            for mode, want in ((0, plain), (1, group)):
                planes = torch.full((slices, M, N), -7, dtype=torch.int32, device=gpu)
                if mode:
                    check(lib.qs_w4a8_per_group_gemm_planes(a.data_ptr(), w.data_ptr(), z.data_ptr(), s.data_ptr(), planes.data_ptr(), M, N, K, st), "planes")
                else:
                    check(lib.qs_w4a8_per_chn_gemm_planes(a.data_ptr(), w.data_ptr(), planes.data_ptr(), M, N, K, st), "planes")
                assert np.array_equal(planes.sum(0).cpu().numpy(), want)
        finally:
            lib.qs_set_gemm_variant(-1)


def test_what_loses_more_than_an_eighth_is_not_taken(gpu):
    A, W = torch.zeros((13, 1152), dtype=torch.int8, device=gpu), torch.zeros((256, 576), dtype=torch.int8, device=gpu)
    lib.qs_set_gemm_variant(4111)                                                           # 18 stages, 8 groups: three rounds for two and a quarter
    try:
        with pytest.raises(RuntimeError):
            acc = torch.empty((13, 256), dtype=torch.int32, device=gpu)
            check(lib.qs_w4a8_per_chn_gemm_acc(A.data_ptr(), W.data_ptr(), acc.data_ptr(), 13, 256, 1152, torch.cuda.current_stream().cuda_stream), "acc")
    finally:
        lib.qs_set_gemm_variant(-1)
