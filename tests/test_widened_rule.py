"""Which per-group products of many tokens ask for scratch (qs_w4a8_per_group_scratch_bytes) and what their entries refuse, without a GPU.  Every shape was measured on both
sides (figures beside the rule)."""
import pytest

from qserve_amd._lib import lib

SLOWER = [(1025, 256, 16384), (4096, 512, 8192), (2048, 1024, 4096), (1300, 1536, 4096), (2048, 1024, 16384),                # one round of channel pairs
          (1300, 2816, 1536),                                                                                                  # two, a short reduction
          (1600, 4096, 1024), (2048, 4096, 1536), (1025, 6144, 1024),                                                          # one round of 128-token tiles, the same
          (800, 2560, 8192), (516, 3840, 5888), (662, 3072, 17152),                                                            # 32-token workgroups of the ring kernel
          (1000, 29696, 2560), (972, 31744, 1024), (906, 31744, 1408)]                                                         # two full rounds of four-wave tiles
FASTER = [(6000, 512, 8192), (4096, 1024, 4096), (1600, 1536, 4096), (1025, 2048, 2048), (1025, 2816, 2048), (4096, 2048, 2048), (1300, 6144, 1024), (800, 5120, 5120),
          (5331, 12288, 4096), (8192, 57344, 8192), (300, 22016, 4096)]


@pytest.mark.parametrize("M, N, K", SLOWER)
def test_where_the_plain_entry_is_the_faster_one(M, N, K):
    assert lib.qs_w4a8_per_group_scratch_bytes(M, N, K) == 0


@pytest.mark.parametrize("M, N, K", FASTER)
def test_where_the_widened_weights_are(M, N, K):
    assert lib.qs_w4a8_per_group_scratch_bytes(M, N, K) == N * K


def test_the_scratch_and_the_grid_are_bounded():
    assert lib.qs_w4a8_per_group_scratch_bytes(2048, 65536, 8192) == 512 << 20
    assert lib.qs_w4a8_per_group_scratch_bytes(2048, 65792, 8192) == 0
    assert lib.qs_w4a8_per_group_scratch_bytes(2048, 32 * 65528, 128) == 32 * 65528 * 128 and lib.qs_w4a8_per_group_scratch_bytes(2048, 32 * 65536, 128) == 0


P256 = 256                                                           # an address that nothing reads: both calls are refused before a launch


def test_what_the_plain_entry_refuses_stays_refused():
    M, N, K = 800, 5120, 4352                                        # the ring kernel, which reads channel scales in pairs
    ops = [P256] * 4
    for fn, tail in ((lib.qs_w4a8_per_group_gemm, ()), (lib.qs_w4a8_per_group_gemm_scratch, (P256, N * K))):
        assert fn(*ops, P256 + 2, P256, P256, M, N, K, *tail, None) == -1 and b"4-byte" in lib.qs_last_error()
    M, N, K = 1300, 4096, 1024                                       # channel pairs, which have no activation epilogue
    for fn, tail in ((lib.qs_w4a8_per_group_gemm_silu_mul, ()), (lib.qs_w4a8_per_group_gemm_silu_mul_scratch, (P256, N * K))):
        assert fn(*ops, P256, P256, P256, None, M, N, K, *tail, None) == -1 and b"tmp" in lib.qs_last_error()
