"""Which per-channel products of prompts run as two launches (qs_w4a8_per_chn_gemm_rounds; no GPU)."""
import pytest

from qserve_amd._lib import lib
from qserve_amd.plan import gemm_plan
from test_gemm_rounds_gpu import FIRST, first_tokens


def _args(at=256, scales=256):
    return at, at, scales, scales, scales, scales, at       # (addresses: looked at, not read)


@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("M, N, K", list(FIRST))
def test_the_first_launch(M, N, K, silu):
    first = first_tokens(_args(), silu, M, N, K)
    assert first == FIRST[M, N, K]
    if first:
        tile = gemm_plan(M, N, K)["tile_tokens"]
        rounds = -(-M // tile) * (N // 256) // 256
        assert first % tile == 0 and first // tile * (N // 256) <= 256 * rounds < (first // tile + 1) * (N // 256)      # as many whole tiles of tokens as the rounds hold


@pytest.mark.parametrize("args", [_args(scales=258), _args(at=264), (0, *_args()[1:])])
def test_arguments_that_keep_to_one_launch(args):
    assert first_tokens(args, False, 4352, 4096, 4096) == 0


def test_a_chosen_variant_keeps_to_one_launch():
    assert first_tokens(_args(), False, 4352, 4096, 4096) == 4096
    lib.qs_set_gemm_variant(4003)
    try:
        assert first_tokens(_args(), False, 4352, 4096, 4096) == 0
    finally:
        lib.qs_set_gemm_variant(-1)
    assert first_tokens(_args(), False, 4352, 4096, 4096) == 4096
