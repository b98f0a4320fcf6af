"""Which per-group products of many tokens ask for scratch (qs_w4a8_per_group_scratch_bytes), without a GPU.  Every shape was measured on both
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
