"""Scratch for widened weights that the allocator has no memory for: the product goes without, and the allocator is left alone for a while."""
import types

import pytest
import torch

from qserve_amd.backend import _util

SHAPE = (1300, 4096, 1024)


def test_a_device_without_memory_is_not_asked_for_every_product(monkeypatch):
    asked = []

    def empty(size, **kw):
        asked.append(size[0])
        if len(asked) in (1, 2):
            raise torch.OutOfMemoryError("none")
        return size

    monkeypatch.setattr(_util.torch, "empty", empty)
    monkeypatch.setattr(_util, "_without", {})
    first, other = (types.SimpleNamespace(device=torch.device("cuda", i)) for i in (0, 1))
    assert all(_util.widened_scratch(*SHAPE, first) is None for _ in range(_util.WITHOUT_SCRATCH + 1)) and len(asked) == 1
    assert _util.widened_scratch(*SHAPE, other) is None and len(asked) == 2                       # (another device has its own count)
    assert _util.widened_scratch(*SHAPE, first) == (4096 * 1024,) and _util.widened_scratch(*SHAPE, first) == (4096 * 1024,)
    assert _util.widened_scratch(256, 4096, 1024, first) is None and len(asked) == 4


@pytest.mark.gpu
@pytest.mark.parametrize("compiled", [False, True], ids=["mirror", "extension"])
def test_products_without_memory_for_scratch(gpu, compiled, monkeypatch):
    if compiled:
        import qserve_backend_ext
        op = qserve_backend_ext.qgemm_w4a8_per_group
    else:
        import qserve_backend.qgemm_w4a8_per_group as op
        monkeypatch.setattr(_util, "_without", {})
    M, N, K = 1300, 24576, 1024                                      # (24 MiB: a segment of its own)
    g = torch.Generator(device=gpu).manual_seed(3)
    X = torch.randint(-128, 128, (M, K), dtype=torch.int8, device=gpu, generator=g)
    W = torch.randint(-128, 128, (N, K // 2), dtype=torch.int8, device=gpu, generator=g)
    s8 = torch.randint(3, 10, (K // 128, N), dtype=torch.int8, device=gpu, generator=g)
    z8, ws, sa = (-(8 * s8.int())).to(torch.int8), torch.rand(N, device=gpu, generator=g).half() * 2e-3, torch.rand(M, device=gpu, generator=g).half() * 1e-2
    assert _util.lib.qs_w4a8_per_group_scratch_bytes(M, N, K) == N * K
    outs = [torch.zeros((M, N), dtype=torch.float16, device=gpu) for _ in range(10)]
    op.gemm_forward_cuda(X, W, z8, s8, ws, sa, outs[0])
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 20)) / total)
    try:
        held = []                                                    # (what earlier tests left free inside segments of theirs)
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                held.append(torch.empty(N * K, dtype=torch.uint8, device=gpu))
        before = torch.cuda.memory_stats()["num_ooms"]
        for out in outs[1:]:
            op.gemm_forward_cuda(X, W, z8, s8, ws, sa, out)
        assert torch.cuda.memory_stats()["num_ooms"] - before == 1
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert all(torch.equal(outs[0].view(torch.int16), out.view(torch.int16)) for out in outs[1:])
