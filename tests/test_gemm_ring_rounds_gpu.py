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
