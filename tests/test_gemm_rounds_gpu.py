"""Per-channel products of prompts in two launches where the last round of tiles is mostly empty: the bits of one launch."""
import ctypes as C

import pytest
import torch

from qserve_amd.backend._util import lib, stream
from qserve_amd.decode import W4A8Linear

pytestmark = pytest.mark.gpu


# (tokens, channels, reduction) -> tokens of the first of two launches, 0: one launch
FIRST = {
    (4097, 4096, 2048): 4096, (4352, 4096, 2048): 4096, (6143, 4096, 2048): 4096, (6144, 4096, 2048): 4096,       # 256-token tiles, one round and a part
    (2049, 4096, 2048): 2048, (2300, 4096, 2048): 2048, (2560, 4096, 2176): 2048,                                 # 128-token tiles
    (2817, 6144, 2048): 2560, (5633, 6144, 4096): 5376, (8192, 4096, 2048): 0, (8193, 4096, 2048): 8192,          # rounds that the channels do not divide; none over
    (577, 28672, 2048): 512, (1281, 28672, 2048): 0, (3585, 28672, 2048): 0, (330, 22016, 2048): 256,             # many channels: others of more than a round
    (4100, 4096, 11008): 4096, (4352, 4096, 14336): 4096, (4352, 4096, 1024): 0,                                  # long reductions, too short a one
    (20000, 512, 2048): 0, (33300, 512, 2048): 32768, (9000, 1792, 2176): 0, (4500, 4096, 2304): 4096}            # few channels, others in 128-channel pairs or by split-K


def first_tokens(args, silu, M, N, K):
    first = C.c_int(-1)
    assert lib.qs_w4a8_per_chn_gemm_rounds(*args, int(silu), M, N, K, C.byref(first)) == 0
    return first.value


@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("offset", [0, 1])                  # (1: scales that start on 2 bytes stay with the tiles)
@pytest.mark.parametrize("M, N, K", list(FIRST))
def test_two_launches(M, N, K, offset, silu):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    if silu and N < 6144:
        pytest.skip("plain there")
    g = torch.Generator(device="cuda").manual_seed(M)
    lin = W4A8Linear(N, K, -1, "cuda", g)
    x = torch.randint(-127, 128, (M, K), dtype=torch.int8, device="cuda", generator=g)
    half = lambda n: (torch.rand(n + offset, device="cuda", generator=g) * 0.002).half()[offset:]                                # noqa: E731
    sa, ss, ws, wz = half(M), half(M), half(N), half(N)
    width = N // 2 if silu else N
    tmp = torch.empty((M, N), dtype=torch.float16, device="cuda") if silu else None

    def run(two):
        out = torch.full((M + 1, width), 7.0, dtype=torch.float16, device="cuda")
        args = (x.data_ptr(), lin.qweight.data_ptr(), ws.data_ptr(), sa.data_ptr(), wz.data_ptr(), ss.data_ptr(), out.data_ptr())
        assert first_tokens(args, silu, M, N, K) == (FIRST[M, N, K] if two else 0)
        rc = lib.qs_w4a8_per_chn_gemm_silu_mul(*args, tmp.data_ptr(), M, N, K, stream()) if silu else lib.qs_w4a8_per_chn_gemm(*args, M, N, K, stream())
        assert rc == 0
        torch.cuda.synchronize()
        assert (out[M] == 7).all()
        return out[:M]
    out = run(offset == 0)
    lib.qs_set_gemm_variant(4003)      # (any variant keeps to one launch; this one says nothing about tiles)
    try:
        ref = run(False)
    finally:
        lib.qs_set_gemm_variant(-1)
    assert torch.equal(out, ref)
