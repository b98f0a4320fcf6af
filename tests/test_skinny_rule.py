"""Which products of few rows go to the kernel that streams the weight: pairs of measured times on either side of the rule's lines."""
import pytest

from qserve_amd.layers.ops import _heads_stream, _prompt_splits, _skinny


# rows, N, K where the vendor's product is the faster one by more than the runs differ
@pytest.mark.parametrize("T, N, K", [(1, 64, 8192), (16, 64, 6144), (33, 64, 7168), (17, 1024, 8192), (64, 1024, 6144), (1, 8192, 8192), (16, 8192, 8192),
                                     (1, 128256, 4096), (16, 128256, 4096), (1, 152064, 8192), (16, 152064, 8192), (1, 32000, 8192), (1, 16384, 16384), (16, 4096, 16384),
                                     (16, 16384, 5120), (16, 4608, 5120), (32, 4608, 5120), (32, 16384, 2048), (32, 14336, 2048), (17, 9216, 3072), (33, 4096, 3072),
                                     (33, 8192, 4096), (64, 32000, 2048), (32, 64, 28672), (65, 2048, 2048)])
def test_left_to_the_vendor(T, N, K):
    assert not _skinny(T, N, K)


@pytest.mark.parametrize("T, N, K", [(1, 16, 2048), (64, 64, 2048), (16, 64, 4096), (64, 1024, 4096), (1, 512, 64), (16, 32000, 4096), (32, 32000, 2048), (16, 128256, 2048),
                                     (32, 8192, 2048), (32, 6144, 4096), (64, 6144, 2048), (64, 2048, 4096), (16, 11008, 4096), (16, 4096, 11008), (32, 4096, 5120),
                                     (16, 8192, 14336), (16, 5120, 13824), (64, 2048, 5632), (64, 4096, 2752), (16, 2048, 5632),
                                     (17, 3072, 5632), (16, 27648, 5120), (16, 512, 11008), (17, 1024, 11008), (33, 1024, 11008), (16, 2048, 18944)])
def test_streamed(T, N, K):
    assert _skinny(T, N, K)


@pytest.mark.parametrize("heads, K, N, takes", [(16, 128, 512, True), (65535, 32, 32, True), (65536, 32, 32, False), (1, 65536, 32768, False), (1, 32, 2 ** 26 - 32, True),
                                                (4, 48, 64, False), (4, 64, 40, False)])
def test_products_per_head_that_the_kernel_takes(heads, K, N, takes):
    import torch
    from qserve_amd.layers.ops import HipOps
    x, w = torch.empty(2, heads, K, dtype=torch.bfloat16, device="meta"), torch.empty(heads, K, N, dtype=torch.bfloat16, device="meta")
    assert HipOps._head_products_fit(None, 2, x, w, K) is takes


def test_the_kernel_is_left_out_where_torch_itself_has_to_be_called():
    import torch
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode
    from qserve_amd.layers.ops import _called_plainly
    x, seen = torch.ones(2, 3), []
    note = lambda t: (seen.append(_called_plainly()), t * 2)[1]                                  # noqa: E731
    assert _called_plainly()
    torch.vmap(note)(x)
    torch.func.jvp(note, (x,), (x,))
    torch.jit.trace(note, (x,), check_trace=False)
    with forward_ad.dual_level():
        note(x)
    with TorchDispatchMode():
        seen.append(_called_plainly())
    assert len(seen) == 5 and not any(seen) and _called_plainly()


def test_products_per_head_are_left_to_torch_where_it_has_to_be_called():
    import torch
    from qserve_amd.layers.ops import HipOps
    x, w, seen = torch.ones(2, 3, 32).bfloat16(), torch.ones(3, 32, 64).bfloat16(), []
    fits = lambda x, w: HipOps._head_products_fit(None, 2, x, w, 32)                             # noqa: E731
    assert fits(x, w)
    assert not fits(x, w.clone().requires_grad_()) and not fits(x.clone().requires_grad_(), w)
    with torch.no_grad():
        assert fits(x, w.clone().requires_grad_())
    torch.vmap(lambda v: (seen.append(fits(x, v)), v)[1])(torch.stack([w, w]))
    torch.func.jvp(lambda v: (seen.append(fits(x, v)), v)[1], (w,), (w,))
    assert seen == [False, False]


# rows, heads, K, N
@pytest.mark.parametrize("T, H, K, N, takes", [(1, 16, 512, 128, True), (64, 16, 512, 128, True), (64, 128, 512, 128, True), (1, 32, 192, 1536, True), (16, 16, 1536, 192, True),
                                               (1, 64, 1024, 128, False), (1, 64, 512, 512, False), (64, 128, 1536, 192, False), (64, 128, 768, 128, False),
                                               (33, 1, 2048, 128, False), (16, 32, 2048, 512, False)])
def test_products_per_head_that_the_kernel_is_faster_at(T, H, K, N, takes):
    assert _heads_stream(T, H, K, N) is takes


# workgroups without a cut, keys, tokens, heads, rank, wide rows: splits whose time is within a few per cent of the best
@pytest.mark.parametrize("groups, span, T, H, rank, wide, good", [(256, 256, 2048, 16, 128, False, {1}), (256, 128, 2048, 16, 128, False, {1}), (128, 128, 512, 32, 128, False, {1}),
                                                                  (192, 256, 2048, 12, 128, False, {1}), (256, 512, 4096, 8, 128, False, {1}), (64, 4096, 512, 16, 128, False, {6, 7, 8}),
                                                                  (1, 4000, 8, 16, 512, True, {24, 32}), (128, 1024, 1024, 16, 512, True, {2}), (512, 4096, 4096, 16, 512, True, {1}),
                                                                  (8, 64, 64, 16, 512, True, {1}), (64, 1000, 256, 16, 512, True, {4}), (1, 2, 2, 1, 128, False, {1})])
def test_cuts_of_a_prompts_keys(groups, span, T, H, rank, wide, good):
    assert _prompt_splits(groups, span, 8 * T * H * rank, wide) in good
