"""Helpers shared by the `qserve_backend` mirror modules: tensor -> device pointer lowering and checks."""
import torch

from .._lib import check, lib  # noqa: F401  (re-exported)


def ptr(t):
    return 0 if t is None else t.data_ptr()


def stream():
    """Current HIP stream as an integer handle (the reference GEMMs use the legacy default stream and the
    attention ops the current stream; the engine never switches streams, so 'current' is equivalent and
    makes the ops capturable in a hipGraph)."""
    return torch.cuda.current_stream().cuda_stream


class guard:
    """Device guard (the reference wraps its attention launch in at::cuda::CUDAGuard, fused_attention.cpp:203; the
    library's per-device scratch and the launch itself follow the CURRENT device): make the tensor's device current for
    the duration of the call.  One cached current_device() query when the device already matches."""
    __slots__ = ("idx", "prev")

    def __init__(self, t):
        self.idx = t.device.index

    def __enter__(self):
        self.prev = torch.cuda.current_device()
        if self.idx is not None and self.prev != self.idx:
            torch.cuda.set_device(self.idx)
        return self

    def __exit__(self, *exc):
        if self.idx is not None and self.prev != self.idx:
            torch.cuda.set_device(self.prev)
        return False


def on_device(t):
    return t.is_cuda


def expect(t, dtype, name, contiguous=True):
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{name} must be a torch.Tensor")
    if t.dtype != dtype:
        # the reference's data_ptr<T>() throws on a dtype mismatch
        raise RuntimeError(f"expected scalar type {dtype} for {name} but found {t.dtype}")
    if not on_device(t):
        raise RuntimeError(f"{name} must be on CUDA")   # wording of the reference's CHECK_DEVICE
    if contiguous and not t.is_contiguous():
        raise RuntimeError(f"{name} must be contiguous")


# A device that had no memory for the scratch is not asked again for this many products: every such request makes torch's allocator give back what it holds.
WITHOUT_SCRATCH = 63
_without = {}                       # device -> products left (a count that threads lose costs a request more or less)


def widened_scratch(M, N, K, like):
    """Scratch for a per-group product of many tokens (include/qserve_amd.h, qs_w4a8_per_group_scratch_bytes), or None: the product needs none - a decode
    step is not asked -, or there is no memory left for it."""
    if M <= 256:
        return None
    need = lib.qs_w4a8_per_group_scratch_bytes(M, N, K)
    if need <= 0:
        return None
    left = _without.get(like.device, 0)
    if left:
        _without[like.device] = left - 1
        return None
    try:
        return torch.empty((need,), dtype=torch.uint8, device=like.device)
    except torch.OutOfMemoryError:
        _without[like.device] = WITHOUT_SCRATCH
        return None
